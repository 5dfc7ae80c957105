// Native half of ullm_amd/attention.py: argument checks, output and scratch
// allocation and the C-ABI calls of the per-token and per-prompt entry points.
//
// A decode step is launch-bound: the kernels of one layer take 6 to 20 us and
// the host has to queue them faster than that.  Host time of one call, us,
// through ctypes and here: attn_decode 12.7 -> 7.2 (two launches; ctypes spent
// 2.9 on the current stream, 1.4 on the output, the rest on arguments),
// GpuAttention.forward 28.7 -> 6.7 (three launches -> the fused step's two) and
// forward_proj 30.5 -> 10.6 (three on both sides).  Functions take positional arguments only
// (METH_FASTCALL); attention.py holds the signatures, defaults and documentation.
// Nothing is kept between calls.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <climits>
#include <cmath>
#include <optional>

#include "../../../include/ullm_hip.h"

namespace {

PyObject *g_error;  // UllmHipError, set once by attention.py

// A failed check or call: UllmHipError(code, message).
struct Fail {
    int code;
    std::string msg;
};
[[noreturn]] void fail(int code, std::string msg) { throw Fail{code, std::move(msg)}; }
[[noreturn]] void invalid(const char *msg) { fail(ULLM_HIP_E_INVALID, msg); }
struct PyRaised {};  // a Python exception is already set
[[noreturn]] void raise(PyObject *type, const char *msg) {
    PyErr_SetString(type, msg);
    throw PyRaised{};
}

// ---- arguments ----
struct Args {
    PyObject *const *a;
    const at::Tensor &t(int i) const {
        if (!THPVariable_Check(a[i])) raise(PyExc_TypeError, "expected a tensor");
        return THPVariable_Unpack(a[i]);
    }
    const at::Tensor *ot(int i) const { return none(i) ? nullptr : &t(i); }
    bool none(int i) const { return a[i] == Py_None; }
    int64_t i64(int i) const {
        PyObject *n = PyNumber_Index(a[i]);
        if (!n) throw PyRaised{};
        const long long v = PyLong_AsLongLong(n);
        Py_DECREF(n);
        if (v == -1 && PyErr_Occurred()) throw PyRaised{};
        return v;
    }
    int i32(int i) const {
        const int64_t v = i64(i);
        if (v != (int)v) raise(PyExc_OverflowError, "integer argument out of range");
        return (int)v;
    }
    // A window; one past every position (2^31 and more) is none.
    int window(int i) const {
        const int64_t v = i64(i);
        return v > INT_MAX || v < 0 ? 0 : (int)v;
    }
    double f(int i) const {
        const double v = PyFloat_AsDouble(a[i]);
        if (v == -1 && PyErr_Occurred()) throw PyRaised{};
        return v;
    }
    bool truth(int i) const {
        const int v = PyObject_IsTrue(a[i]);
        if (v < 0) throw PyRaised{};
        return v;
    }
};

int dt(const at::Tensor &t) {
    switch (t.scalar_type()) {
        case at::kFloat: return ULLM_DT_F32;
        case at::kHalf: return ULLM_DT_F16;
        case at::kBFloat16: return ULLM_DT_BF16;
        default:
            fail(ULLM_HIP_E_UNSUPPORTED, std::string("dtype ") + c10::toString(t.scalar_type()) + " not supported");
    }
}
void *ptr(const at::Tensor *t) { return t ? t->data_ptr() : nullptr; }
const float *fptr(const at::Tensor *t) { return (const float *)ptr(t); }
void need_cuda(std::initializer_list<const at::Tensor *> ts) {
    for (const at::Tensor *t : ts)
        if (t && !t->is_cuda()) invalid("tensors must live on the GPU");
}
bool f32_rows(const at::Tensor &t) { return t.scalar_type() == at::kFloat && t.is_contiguous(); }

// The call's stream: the caller's (any object with .cuda_stream) or torch's
// current one.
struct Stream {
    void *s;
    bool given;
    Stream(const Args &a, int i) : given(!a.none(i)) {
        if (!given) {
            s = (void *)c10::hip::getCurrentHIPStream().stream();
            return;
        }
        PyObject *v = PyObject_GetAttrString(a.a[i], "cuda_stream");
        if (!v) throw PyRaised{};
        s = PyLong_AsVoidPtr(v);
        Py_DECREF(v);
        if (!s && PyErr_Occurred()) throw PyRaised{};
    }
    // Scratch of one call, from this stream's own memory: what held the block
    // before and what takes it next are in order with the call, whichever
    // stream is torch's current one.
    at::Tensor scratch(const at::Tensor &like, int64_t bytes) const {
        const auto dev = like.device().index();
        struct Current {
            c10::hip::HIPStream was;
            explicit Current(c10::DeviceIndex d) : was(c10::hip::getCurrentHIPStream(d)) {}
            ~Current() { c10::hip::setCurrentHIPStream(was); }
        };
        std::optional<Current> back;
        if (given) {
            back.emplace(dev);
            c10::hip::setCurrentHIPStream(c10::hip::getStreamFromExternal((hipStream_t)s, dev));
        }
        return at::empty({bytes}, like.options().dtype(at::kByte));
    }
    // Scratch that a call can do without: undefined where memory has run out.
    at::Tensor scratch_if_any(const at::Tensor &like, int64_t bytes) const {
        if (bytes)
            try {
                return scratch(like, bytes);
            } catch (const c10::OutOfMemoryError &) {
            }
        return at::Tensor();
    }
};

template <class F>
void call(F &&f) {
    PyThreadState *ts = PyEval_SaveThread();
    const int rc = f();
    PyEval_RestoreThread(ts);
    if (rc != ULLM_HIP_OK) fail(rc, ullm_hip_last_error());
}

at::Tensor out_or(const at::Tensor *out, at::IntArrayRef shape, const at::Tensor &like,
                  at::ScalarType st = at::kFloat) {
    return out ? *out : at::empty(shape, like.options().dtype(st));
}

// ---- the entry points ----
at::Tensor decode(const Args &a) {
    // q k v seq_lens max_len n_kv window scale kv_stride seq_stride out ws stream
    const at::Tensor &q = a.t(0), &k = a.t(1), &v = a.t(2), &lens = a.t(3);
    if (q.dim() != 3) raise(PyExc_ValueError, "q must be [B, n_head, head_dim]");
    const int B = (int)q.size(0), H = (int)q.size(1), D = (int)q.size(2), max_len = a.i32(4), hk = a.i32(5),
              win = a.window(6);
    need_cuda({&q, &k, &v, &lens});
    if (!f32_rows(q)) invalid("q must be contiguous f32 [B, n_head, head_dim]");
    if (lens.scalar_type() != at::kInt || lens.numel() != B) invalid("seq_lens must be int32 [B]");
    const float scale = a.none(7) ? (float)(1.0 / std::sqrt((double)D)) : (float)a.f(7);
    const int64_t kvs = a.none(8) ? (int64_t)hk * D : a.i64(8), ss = a.i64(9);
    const Stream st(a, 12);
    const at::Tensor out = out_or(a.ot(10), {B, H, D}, q);
    at::Tensor ws;
    if (!a.none(11)) ws = a.t(11);
    else ws = st.scratch(q, std::max<int64_t>(256, ullm_hip_decode_workspace_bytes(B, H, hk, D, max_len, win)));
    const int kd = dt(k);
    call([&] {
        return ullm_hip_attn_decode(fptr(&q), k.data_ptr(), v.data_ptr(), kd, kvs, ss, (const int32_t *)lens.data_ptr(),
                                    max_len, win, B, H, hk, D, scale, (float *)out.data_ptr(), ws.data_ptr(),
                                    ws.numel(), st.s);
    });
    return out;
}

at::Tensor decode_paged(const Args &a) {
    // q k_pages v_pages block_table seq_lens max_len n_kv window scale out ws stream
    const at::Tensor &q = a.t(0), &k = a.t(1), &v = a.t(2), &tab = a.t(3), &lens = a.t(4);
    if (q.dim() != 3) raise(PyExc_ValueError, "q must be [B, n_head, head_dim]");
    const int B = (int)q.size(0), H = (int)q.size(1), D = (int)q.size(2), max_len = a.i32(5), hk = a.i32(6),
              win = a.window(7);
    need_cuda({&q, &k, &v, &tab, &lens});
    if (!f32_rows(q)) invalid("q must be contiguous f32 [B, n_head, head_dim]");
    if (k.dim() != 3 || k.sizes() != v.sizes() || !k.is_contiguous() || !v.is_contiguous())
        invalid("k_pages/v_pages must be contiguous [n_pages, page_size, kv_stride]");
    if (tab.scalar_type() != at::kInt || tab.dim() != 2 || tab.size(0) != B || !tab.is_contiguous())
        invalid("block_table must be contiguous int32 [B, table_stride]");
    if (lens.scalar_type() != at::kInt || lens.numel() != B) invalid("seq_lens must be int32 [B]");
    const float scale = a.none(8) ? (float)(1.0 / std::sqrt((double)D)) : (float)a.f(8);
    const Stream st(a, 11);
    const at::Tensor out = out_or(a.ot(9), {B, H, D}, q);
    at::Tensor ws;
    if (!a.none(10)) ws = a.t(10);
    else ws = st.scratch(q, std::max<int64_t>(256, ullm_hip_paged_decode_workspace_bytes(B, H, hk, D, max_len, win)));
    const int kd = dt(k);
    call([&] {
        return ullm_hip_attn_decode_paged(fptr(&q), k.data_ptr(), v.data_ptr(), kd, k.size(2), (int)k.size(1),
                                          (int)k.size(0), (const int32_t *)tab.data_ptr(), (int)tab.size(1),
                                          (const int32_t *)lens.data_ptr(), max_len, win, B, H, hk, D, scale,
                                          (float *)out.data_ptr(), ws.data_ptr(), ws.numel(), st.s);
    });
    return out;
}

// The norm, bias and RoPE arguments shared by the appends and projections.
struct Prep {
    const at::Tensor &cs;
    int H, hk, D, rd, neox;
    const at::Tensor *qn, *kn;
    float eps;
    const at::Tensor *qb, *kb, *vb;
    // rope_cs n_head n_kv head_dim rotary_dim neox q_norm k_norm eps q_bias k_bias v_bias from argument i
    static constexpr int N = 12;
    Prep(const Args &a, int i)
        : cs(a.t(i)), H(a.i32(i + 1)), hk(a.i32(i + 2)), D(a.i32(i + 3)), rd(a.none(i + 4) ? D : a.i32(i + 4)),
          neox(a.truth(i + 5)), qn(a.ot(i + 6)), kn(a.ot(i + 7)), eps((float)a.f(i + 8)), qb(a.ot(i + 9)),
          kb(a.ot(i + 10)), vb(a.ot(i + 11)) {}
};
at::ScalarType dtype_arg(const Args &a, int i) {
    if (a.none(i)) return at::kFloat;
    if (!THPDtype_Check(a.a[i])) raise(PyExc_TypeError, "q_dtype must be a torch.dtype");
    return ((THPDtype *)a.a[i])->scalar_type;
}

void append_call(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v, const Prep &p, int rows,
                 int64_t start, const at::Tensor &qo, void *kc, void *vc, int kd, int64_t kvs, void *s) {
    const int qd = dt(qo);
    call([&] {
        return ullm_hip_qkv_append(fptr(&q), fptr(&k), fptr(&v), fptr(p.qb), fptr(p.kb), fptr(p.vb), fptr(p.qn),
                                   fptr(p.kn), p.eps, fptr(&p.cs), (int)p.cs.size(0), p.neox, p.rd, rows, (int)start,
                                   p.H, p.hk, p.D, qo.data_ptr(), qd, kc, vc, kd, kvs, s);
    });
}

at::Tensor append(const Args &a) {
    // q k v k_cache v_cache start_pos <Prep> q_out q_dtype kv_stride stream
    const at::Tensor &q = a.t(0), &k = a.t(1), &v = a.t(2), &kc = a.t(3), &vc = a.t(4);
    const int start = a.i32(5);
    const Prep p(a, 6);
    constexpr int R = 6 + Prep::N;
    need_cuda({&q, &k, &v, &kc, &vc, &p.cs});
    if (!f32_rows(q) || !f32_rows(k) || !f32_rows(v)) invalid("q/k/v must be contiguous f32");
    const Stream st(a, R + 3);
    const int rows = (int)q.size(0);
    const at::Tensor qo = out_or(a.ot(R), {rows, (int64_t)p.H * p.D}, q, dtype_arg(a, R + 1));
    append_call(q, k, v, p, rows, start, qo, kc.data_ptr(), vc.data_ptr(), dt(kc),
                a.none(R + 2) ? (int64_t)p.hk * p.D : a.i64(R + 2), st.s);
    return qo;
}

at::Tensor append_paged(const Args &a) {
    // q k v k_pages v_pages positions block_table <Prep> q_out q_dtype stream
    const at::Tensor &q = a.t(0), &k = a.t(1), &v = a.t(2), &kp = a.t(3), &vp = a.t(4), &pos = a.t(5), &tab = a.t(6);
    const Prep p(a, 7);
    constexpr int R = 7 + Prep::N;
    const int rows = (int)q.size(0);
    need_cuda({&q, &k, &v, &kp, &vp, &p.cs, &pos, &tab});
    if (!f32_rows(q) || !f32_rows(k) || !f32_rows(v)) invalid("q/k/v must be contiguous f32");
    if (kp.dim() != 3 || kp.sizes() != vp.sizes()) invalid("k_pages/v_pages must be [n_pages, page_size, kv_stride]");
    if (pos.scalar_type() != at::kInt || pos.numel() != rows) invalid("positions must be int32 [rows]");
    if (tab.scalar_type() != at::kInt || tab.dim() != 2 || tab.size(0) != rows || !tab.is_contiguous())
        invalid("block_table must be contiguous int32 [rows, table_stride]");
    const Stream st(a, R + 2);
    const at::Tensor qo = out_or(a.ot(R), {rows, (int64_t)p.H * p.D}, q, dtype_arg(a, R + 1));
    const int qd = dt(qo), kd = dt(kp);
    call([&] {
        return ullm_hip_qkv_append_paged(
            fptr(&q), fptr(&k), fptr(&v), fptr(p.qb), fptr(p.kb), fptr(p.vb), fptr(p.qn), fptr(p.kn), p.eps,
            fptr(&p.cs), (int)p.cs.size(0), p.neox, p.rd, rows, (const int32_t *)pos.data_ptr(), p.H, p.hk, p.D,
            qo.data_ptr(), qd, kp.data_ptr(), vp.data_ptr(), kd, kp.size(2), (int)kp.size(1), (int)kp.size(0),
            (const int32_t *)tab.data_ptr(), (int)tab.size(1), st.s);
    });
    return qo;
}

// The checks of the projections' x and weights.
void proj_check(const at::Tensor &x, const at::Tensor &wq, const at::Tensor &wk, const at::Tensor &wv, int64_t in_dim,
                const Prep &p) {
    if (!f32_rows(x)) invalid("x must be contiguous f32");
    if (wq.scalar_type() != wk.scalar_type() || wk.scalar_type() != wv.scalar_type())
        invalid("w_q/w_k/w_v must share one dtype");
    const at::Tensor *ws[3] = {&wq, &wk, &wv};
    for (int i = 0; i < 3; i++) {
        const at::Tensor &w = *ws[i];
        const int64_t n = (int64_t)(i ? p.hk : p.H) * p.D;
        if (w.dim() != 2 || w.size(0) != n || w.size(1) != in_dim || !w.is_contiguous()) {
            std::string got;
            for (int64_t d : w.sizes()) got += (got.empty() ? "" : ", ") + std::to_string(d);
            fail(ULLM_HIP_E_INVALID, "weight shape (" + got + ") != (" + std::to_string(n) + ", " +
                                         std::to_string(in_dim) + ")");
        }
    }
}

void proj_call(const at::Tensor &x, const at::Tensor &wq, const at::Tensor &wk, const at::Tensor &wv, int64_t in_dim,
               const Prep &p, int rows, int64_t start, const at::Tensor &qo, void *kc, void *vc, int kd, int64_t kvs,
               const at::Tensor *ws, void *s) {
    const int wd = dt(wq), qd = dt(qo);
    call([&] {
        return ullm_hip_qkv_proj_append(fptr(&x), (int)in_dim, wq.data_ptr(), wk.data_ptr(), wv.data_ptr(), wd,
                                        fptr(p.qb), fptr(p.kb), fptr(p.vb), fptr(p.qn), fptr(p.kn), p.eps, fptr(&p.cs),
                                        (int)p.cs.size(0), p.neox, p.rd, rows, (int)start, p.H, p.hk, p.D,
                                        qo.data_ptr(), qd, kc, vc, kd, kvs, ptr(ws), ws ? ws->nbytes() : 0, s);
    });
}

// One matvec per row (and the workspace of the caller), or one GEMM over the
// rows with its own scratch: x_bits 0 or 16 / 24.  None where the GEMM does not
// take the sizes or has no memory for its scratch.
PyObject *proj(const Args &a) {
    // x w_q w_k w_v k_cache v_cache start_pos x_bits <Prep> q_out q_dtype kv_stride ws stream
    const at::Tensor &x = a.t(0), &wq = a.t(1), &wk = a.t(2), &wv = a.t(3), &kc = a.t(4), &vc = a.t(5);
    const int start = a.i32(6), bits = a.i32(7);
    const Prep p(a, 8);
    constexpr int R = 8 + Prep::N;
    if (x.dim() != 2) raise(PyExc_ValueError, "x must be [rows, in_dim]");
    const int64_t rows = x.size(0), in_dim = x.size(1);
    need_cuda({&x, &wq, &wk, &wv, &kc, &vc, &p.cs});
    proj_check(x, wq, wk, wv, in_dim, p);
    const Stream st(a, R + 4);
    const int wd = dt(wq), kd = dt(kc);
    const int64_t kvs = a.none(R + 2) ? (int64_t)p.hk * p.D : a.i64(R + 2);
    if (rows != (int)rows || in_dim != (int)in_dim) invalid("x: sizes of 2^31 or more");
    size_t need = 0;
    at::Tensor ws;
    if (bits) {
        need = ullm_hip_qkv_gemm_workspace_bytes((int)rows, (int)in_dim, wd, bits, p.H, p.hk, p.D);
        ws = st.scratch_if_any(x, need);
        if (!ws.defined()) Py_RETURN_NONE;
    }
    const at::Tensor qo = out_or(a.ot(R), {rows, (int64_t)p.H * p.D}, x, dtype_arg(a, R + 1));
    if (!bits) {
        proj_call(x, wq, wk, wv, in_dim, p, (int)rows, start, qo, kc.data_ptr(), vc.data_ptr(), kd, kvs,
                  a.ot(R + 3), st.s);
    } else {
        const int qd = dt(qo);
        call([&] {
            return ullm_hip_qkv_gemm_append(
                fptr(&x), (int)in_dim, wq.data_ptr(), wk.data_ptr(), wv.data_ptr(), wd, bits, fptr(p.qb), fptr(p.kb),
                fptr(p.vb), fptr(p.qn), fptr(p.kn), p.eps, fptr(&p.cs), (int)p.cs.size(0), p.neox, p.rd, (int)rows,
                start, p.H, p.hk, p.D, qo.data_ptr(), qd, kc.data_ptr(), vc.data_ptr(), kd, kvs, ws.data_ptr(),
                need, st.s);
        });
    }
    return THPVariable_Wrap(qo);
}

at::Tensor prefill(const Args &a) {
    // q k_cache v_cache n_head n_kv head_dim start_pos window scale kv_stride out stream max_q_bytes
    const at::Tensor &q = a.t(0), &k = a.t(1), &v = a.t(2);
    const int H = a.i32(3), hk = a.i32(4), D = a.i32(5), start = a.i32(6), win = a.window(7);
    const int64_t S = q.size(0), row = (int64_t)H * D;
    need_cuda({&q, &k, &v});
    if (!q.is_contiguous() || q.numel() != S * row) invalid("q must be contiguous [S, n_head*head_dim]");
    if (q.scalar_type() != k.scalar_type() || q.scalar_type() != v.scalar_type()) invalid("q and cache dtypes differ");
    const float scale = a.none(8) ? (float)(1.0 / std::sqrt((double)D)) : (float)a.f(8);
    const int64_t kvs = a.none(9) ? (int64_t)hk * D : a.i64(9);
    const Stream st(a, 11);
    const at::Tensor out = out_or(a.ot(10), {S, row}, q);
    const int qd = dt(q);
    const int64_t step = std::max<int64_t>(1, a.i64(12) / std::max<int64_t>(1, row * (int64_t)q.element_size()));
    for (int64_t r0 = 0; r0 < std::max<int64_t>(S, 1); r0 += step) {
        const int n = (int)std::min(step, S - r0);
        const size_t need = ullm_hip_prefill_workspace_bytes(qd, n, start + (int)r0, win, H, hk, D);
        const at::Tensor ws = st.scratch_if_any(q, need);
        call([&] {
            return ullm_hip_attn_prefill_ws((const char *)q.data_ptr() + r0 * row * q.element_size(), k.data_ptr(),
                                            v.data_ptr(), qd, kvs, n, start + (int)r0, win, H, hk, D, scale,
                                            (float *)out.data_ptr() + r0 * row, ws.defined() ? ws.data_ptr() : nullptr,
                                            need, st.s);
        });
    }
    return out;
}

at::Tensor prefill_paged(const Args &a) {
    // q k_pages v_pages block_table n_head n_kv head_dim start_pos window scale out stream
    const at::Tensor &q = a.t(0), &k = a.t(1), &v = a.t(2), &tab = a.t(3);
    const int H = a.i32(4), hk = a.i32(5), D = a.i32(6), start = a.i32(7), win = a.window(8);
    const int64_t S = q.size(0), row = (int64_t)H * D;
    need_cuda({&q, &k, &v, &tab});
    if (!q.is_contiguous() || q.numel() != S * row) invalid("q must be contiguous [S, n_head*head_dim]");
    if (k.dim() != 3 || k.sizes() != v.sizes() || q.scalar_type() != k.scalar_type())
        invalid("k_pages/v_pages must be [n_pages, page_size, kv_stride] of q's dtype");
    if (tab.scalar_type() != at::kInt || tab.dim() != 1) invalid("block_table must be int32 [table_len]");
    const float scale = a.none(9) ? (float)(1.0 / std::sqrt((double)D)) : (float)a.f(9);
    const Stream st(a, 11);
    const at::Tensor out = out_or(a.ot(10), {S, row}, q);
    const int qd = dt(q);
    const size_t need = ullm_hip_prefill_workspace_bytes(qd, (int)S, start, win, H, hk, D);
    const at::Tensor ws = st.scratch_if_any(q, need);
    call([&] {
        return ullm_hip_attn_prefill_paged_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), qd, k.size(2), (int)k.size(1),
                                              (int)k.size(0), (const int32_t *)tab.data_ptr(), (int)tab.numel(), (int)S,
                                              start, win, H, hk, D, scale, (float *)out.data_ptr(),
                                              ws.defined() ? ws.data_ptr() : nullptr, need, st.s);
    });
    return out;
}

// One decoded token of GpuAttention: the append (from q, k, v) or the fused
// projection (from the hidden state), then attention over the layer's cache.
struct Layer {
    char *k, *v;
    int kd;
    Layer(const at::Tensor &kc, const at::Tensor &vc, int64_t layer) {
        const int64_t n = kc.size(0);
        if (layer < -n || layer >= n) raise(PyExc_IndexError, "layer index out of range");
        if (layer < 0) layer += n;
        k = (char *)kc.data_ptr() + layer * kc.stride(0) * (int64_t)kc.element_size();
        v = (char *)vc.data_ptr() + layer * vc.stride(0) * (int64_t)vc.element_size();
        kd = dt(kc);
    }
};
at::Tensor token(const Args &a) {
    // proj layer pos key_cache val_cache lens ws window scale <Prep> in0..in3 proj_ws
    const bool is_proj = a.truth(0);
    const int64_t layer = a.i64(1);
    const int pos = a.i32(2), win = a.window(7);
    const at::Tensor &kc = a.t(3), &vc = a.t(4), &lens = a.t(5), &ws = a.t(6);
    const float scale = (float)a.f(8);
    const Prep p(a, 9);
    constexpr int R = 9 + Prep::N;
    const at::Tensor &x = a.t(R), &w0 = a.t(R + 1), &w1 = a.t(R + 2);
    const Layer l(kc, vc, layer);
    void *s = (void *)c10::hip::getCurrentHIPStream().stream();
    const int64_t row = (int64_t)p.H * p.D, kvs = (int64_t)p.hk * p.D;
    const at::Tensor *w2 = is_proj ? &a.t(R + 3) : nullptr;
    need_cuda({&x, &w0, &w1, w2, &kc, &vc, &p.cs});
    if (is_proj) proj_check(x, w0, w1, *w2, x.numel(), p);
    else if (!f32_rows(x) || !f32_rows(w0) || !f32_rows(w1)) invalid("q/k/v must be contiguous f32");
    // Append and attention in the attention's two launches, where the shape and
    // the alignment allow it; whatever is refused below is refused there too.
    const auto odd = [](const void *q) { return ((uintptr_t)q & 15) != 0; };
    const size_t need = ullm_hip_decode_token_workspace_bytes(l.kd, pos, win, p.H, p.hk, p.D, p.rd);
    bool fuse = need && ws.numel() >= (int64_t)need && pos < p.cs.size(0) && kvs * (int64_t)kc.element_size() % 16 == 0 &&
                ((int64_t)pos + 1) * kvs * (int64_t)kc.element_size() <= 0x7fff0000LL;
    const void *used[] = {l.k, l.v, ptr(&p.cs), ptr(p.qb), ptr(p.kb), ptr(p.vb), ptr(p.qn), ptr(p.kn), ptr(&x),
                          ptr(&w0), ptr(&w1), ptr(w2)};
    for (const void *q : used)
        fuse = fuse && !odd(q);
    if (is_proj) fuse = fuse && x.numel() >= 8 && x.numel() % 8 == 0;
    // Raw rows projected straight into the position's f32 cache rows: the append
    // takes them in place, the fused launch stores there while others read.
    const int64_t rb = kvs * (int64_t)kc.element_size();
    const auto over = [&](const at::Tensor &t, const char *c) {
        const uintptr_t p = (uintptr_t)t.data_ptr(), r = (uintptr_t)c + pos * rb;
        return p < r + rb && r < p + t.nbytes();
    };
    if (!is_proj)
        for (const at::Tensor *t : {&x, &w0, &w1}) fuse = fuse && !over(*t, l.k) && !over(*t, l.v);
    if (fuse) {
        const float *q = fptr(&x), *k = fptr(&w0), *v = fptr(&w1);
        at::Tensor y;
        if (is_proj) {
            y = at::empty({row + 2 * kvs}, x.options().dtype(at::kFloat));
            const int wd = dt(w0);
            call([&] {
                return ullm_hip_qkv_matvec(fptr(&x), (int)x.numel(), w0.data_ptr(), w1.data_ptr(), w2->data_ptr(), wd,
                                           p.H, p.hk, p.D, (float *)y.data_ptr(), s);
            });
            q = fptr(&y), k = q + row, v = k + kvs;
        }
        const at::Tensor out = at::empty({row}, x.options().dtype(at::kFloat));
        call([&] {
            return ullm_hip_decode_token(q, k, v, fptr(p.qb), fptr(p.kb), fptr(p.vb), fptr(p.qn), fptr(p.kn), p.eps,
                                         fptr(&p.cs), (int)p.cs.size(0), p.neox, pos,
                                         (const int32_t *)lens.data_ptr() + pos - 1, win, p.H, p.hk, p.D, scale, l.k,
                                         l.v, l.kd, kvs, (float *)out.data_ptr(), ws.data_ptr(), ws.numel(), s);
        });
        return out;
    }
    const at::Tensor q = at::empty({1, row}, x.options().dtype(at::kFloat));
    if (is_proj) proj_call(x, w0, w1, *w2, x.numel(), p, 1, pos, q, l.k, l.v, l.kd, kvs, a.ot(R + 4), s);
    else append_call(x, w0, w1, p, 1, pos, q, l.k, l.v, l.kd, kvs, s);
    const at::Tensor out = at::empty({row}, q.options());
    call([&] {
        return ullm_hip_attn_decode(fptr(&q), l.k, l.v, l.kd, kvs, 0, (const int32_t *)lens.data_ptr() + pos, pos + 1,
                                    win, 1, p.H, p.hk, p.D, scale, (float *)out.data_ptr(), ws.data_ptr(), ws.numel(),
                                    s);
    });
    return out;
}

// ---- Python entry ----
template <class F>
PyObject *guard(F &&f) {
    HANDLE_TH_ERRORS
    try {
        return f();
    } catch (const Fail &e) {
        PyObject *x = PyObject_CallFunction(g_error, "is", e.code, e.msg.c_str());
        if (x) {
            PyErr_SetObject(g_error, x);
            Py_DECREF(x);
        }
        return nullptr;
    } catch (const PyRaised &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}
template <at::Tensor (*F)(const Args &), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != N) return PyErr_Format(PyExc_TypeError, "%d arguments expected, %zd given", N, n), nullptr;
    return guard([&] { return THPVariable_Wrap(F(Args{args})); });
}
PyObject *proj_entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 8 + Prep::N + 5) return PyErr_Format(PyExc_TypeError, "%zd arguments given", n), nullptr;
    return guard([&] { return proj(Args{args}); });
}
PyObject *set_error(PyObject *, PyObject *cls) {
    Py_INCREF(cls);
    Py_XSETREF(g_error, cls);
    Py_RETURN_NONE;
}

#define FAST(f) (PyCFunction)(void (*)(void))(PyObject * (*)(PyObject *, PyObject *const *, Py_ssize_t))(f)
PyMethodDef methods[] = {
    {"set_error", set_error, METH_O, nullptr},
    {"decode", FAST((entry<decode, 13>)), METH_FASTCALL, nullptr},
    {"decode_paged", FAST((entry<decode_paged, 12>)), METH_FASTCALL, nullptr},
    {"append", FAST((entry<append, 6 + Prep::N + 4>)), METH_FASTCALL, nullptr},
    {"append_paged", FAST((entry<append_paged, 7 + Prep::N + 3>)), METH_FASTCALL, nullptr},
    {"proj", FAST(proj_entry), METH_FASTCALL, nullptr},
    {"prefill", FAST((entry<prefill, 13>)), METH_FASTCALL, nullptr},
    {"prefill_paged", FAST((entry<prefill_paged, 12>)), METH_FASTCALL, nullptr},
    {"token", FAST((entry<token, 9 + Prep::N + 5>)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_front", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front() { return PyModule_Create(&module); }
