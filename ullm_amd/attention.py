"""Torch-tensor front end of the C ABI, and `GpuAttention`, the attention
part of the reference's `GpuForward` (crates/ullm-metal/src/forward.rs).

Every op here is a thin call into libullm_hip.so, through the native front end
_front.so (argument checks, outputs and scratch, the call; csrc/front/front.cpp);
torch supplies device memory and the current HIP stream and nothing else.  There is no CPU or
PyTorch fallback: without the library or a GPU the calls raise.
"""
from __future__ import annotations

import ctypes as C
import functools
import math
from dataclasses import dataclass
from typing import Optional

import torch

from . import _lib as L

class _NoFront:
    """Stands for the native front end where it does not load: every use raises."""

    def __init__(self, why):
        self._why = why

    def __getattr__(self, name):
        raise ImportError(f"ullm_amd/_front.so does not load ({self._why}): build it with "
                          "`python -m ullm_amd.build` (there is no fallback)")


try:
    from . import _front as _F

    _F.set_error(L.UllmHipError)
except ImportError as e:
    _F = _NoFront(e)

_DT = {torch.float32: L.DT_F32, torch.float16: L.DT_F16, torch.bfloat16: L.DT_BF16}


def _dt(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise L.UllmHipError(L.E_UNSUPPORTED, f"dtype {t.dtype} not supported") from None


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else C.c_void_p(t.data_ptr())


def _stream(stream=None):
    s = torch.cuda.current_stream() if stream is None else stream
    return C.c_void_p(s.cuda_stream)


def _need_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise L.UllmHipError(L.E_INVALID, "tensors must live on the GPU")


def decode_workspace_bytes(batch, n_head, n_kv_head, head_dim, max_len, window=0) -> int:
    return int(L.lib().ullm_hip_decode_workspace_bytes(batch, n_head, n_kv_head, head_dim,
                                                       max_len, window))


def new_decode_workspace(batch, n_head, n_kv_head, head_dim, max_len, window=0, device="cuda"):
    """Workspace for attn_decode (split partials; zeroed only for determinism of
    unused bytes, the kernels write every partial before reading it)."""
    n = max(decode_workspace_bytes(batch, n_head, n_kv_head, head_dim, max_len, window), 256)
    return torch.zeros(n, dtype=torch.uint8, device=device)


def attn_decode(q, k_cache, v_cache, seq_lens, max_len, n_kv_head, *, window=0, scale=None,
                kv_stride=None, seq_stride=0, out=None, workspace=None, stream=None):
    """Single-query GQA decode attention (lib.rs:911-938 / :1180-1208).

    q: [B, n_head, D] f32.  k_cache/v_cache: layer base (f32/f16/bf16) with
    `kv_stride` elements per position (default n_kv_head*D) and `seq_stride`
    between sequences.  seq_lens: int32 [B] on the GPU (= pos + 1).
    """
    return _F.decode(q, k_cache, v_cache, seq_lens, max_len, n_kv_head, window, scale, kv_stride,
                     seq_stride, out, workspace, stream)


def attn_decode_paged(q, k_pages, v_pages, block_table, seq_lens, max_len, n_kv_head, *,
                      window=0, scale=None, out=None, workspace=None, stream=None):
    """Decode attention over a paged KV cache (same result as attn_decode).

    q: [B, n_head, D] f32.  k_pages/v_pages: [n_pages, page_size, kv_stride]
    f16/bf16.  block_table: int32 [B, table_stride] (page of position t of
    sequence b = block_table[b, t // page_size]).  seq_lens: int32 [B].
    """
    return _F.decode_paged(q, k_pages, v_pages, block_table, seq_lens, max_len, n_kv_head, window,
                           scale, out, workspace, stream)


def qkv_append_paged(q, k, v, k_pages, v_pages, rope_cs, positions, block_table, *, n_head,
                     n_kv_head, head_dim, rotary_dim=None, neox=True, q_norm=None, k_norm=None,
                     eps=1e-6, q_bias=None, k_bias=None, v_bias=None, q_out=None, q_dtype=None,
                     stream=None):
    """Append one token per sequence into a paged cache: row r of q/k/v [rows,
    *] f32 is sequence r's token at positions[r] (int32 [rows] on the GPU);
    its K/V rows land in block_table[r, pos // page_size].  Returns q_out."""
    return _F.append_paged(q, k, v, k_pages, v_pages, positions, block_table, rope_cs, n_head,
                           n_kv_head, head_dim, rotary_dim, neox, q_norm, k_norm, eps, q_bias,
                           k_bias, v_bias, q_out, q_dtype, stream)


def attn_prefill_paged(q, k_pages, v_pages, block_table, n_head, n_kv_head, head_dim, *,
                       start_pos=0, window=0, scale=None, out=None, stream=None):
    """Causal prefill of S rows (positions start_pos..) of one sequence whose
    keys live in pages: block_table int32 [table_len] (page of key t =
    block_table[t // page_size]).  q: [S, n_head*head_dim] f16/bf16, or f32
    with f32 pages (head_dim 64, 128 or 256)."""
    return _F.prefill_paged(q, k_pages, v_pages, block_table, n_head, n_kv_head, head_dim,
                            start_pos, window, scale, out, stream)


# Largest q the prefill entry points take in one call (below 2 GiB, and a
# multiple of 16 bytes so every chunk stays 16-byte aligned).
PREFILL_Q_MAX_BYTES = 0x7fff0000


def attn_prefill(q, k_cache, v_cache, n_head, n_kv_head, head_dim, *, start_pos=0, window=0,
                 scale=None, kv_stride=None, out=None, stream=None):
    """Causal prefill attention on MFMA (lib.rs:1061-1087).

    q: [S, n_head*head_dim] in the cache dtype (f16, bf16 or f32); the cache
    already holds positions 0..start_pos+S-1.  Returns [S, n_head*head_dim]
    f32.  A q of PREFILL_Q_MAX_BYTES or more (the kernels address it through
    a 32-bit buffer range) runs as row chunks at increasing start_pos: the
    cache already holds every position, so each chunk's rows see the same
    keys.
    """
    return _F.prefill(q, k_cache, v_cache, n_head, n_kv_head, head_dim, start_pos, window, scale,
                      kv_stride, out, stream, PREFILL_Q_MAX_BYTES)


def rope_table(n_pos: int, rotary_dim: int, theta: float, device="cuda") -> torch.Tensor:
    """(cos, sin) table [n_pos, rotary_dim/2, 2] with the reference formula,
    computed on the host by the library and uploaded."""
    host = torch.empty(n_pos, rotary_dim // 2, 2, dtype=torch.float32)
    L.check(L.lib().ullm_hip_rope_table(C.c_void_p(host.data_ptr()), n_pos, rotary_dim,
                                        float(theta)))
    return host.to(device) if device != "cpu" else host


def qkv_append(q, k, v, k_cache, v_cache, rope_cs, *, start_pos, n_head, n_kv_head, head_dim,
               rotary_dim=None, neox=True, q_norm=None, k_norm=None, eps=1e-6, q_bias=None,
               k_bias=None, v_bias=None, q_out=None, q_dtype=None, kv_stride=None, stream=None):
    """Fused bias + Q/K RMSNorm + RoPE + KV append (lib.rs:1021-1058).

    q: [rows, n_head*D] f32, k/v: [rows, n_kv_head*D] f32.  K/V land in the
    cache at positions start_pos..; returns q_out ([rows, n_head*D], q_dtype).
    """
    return _F.append(q, k, v, k_cache, v_cache, start_pos, rope_cs, n_head, n_kv_head, head_dim,
                     rotary_dim, neox, q_norm, k_norm, eps, q_bias, k_bias, v_bias, q_out, q_dtype,
                     kv_stride, stream)


_proj_ws = {}


@functools.lru_cache(maxsize=256)
def _proj_ws_bytes(rows, n_head, n_kv_head, head_dim):
    return int(L.lib().ullm_hip_qkv_proj_workspace_bytes(rows, n_head, n_kv_head, head_dim))


def proj_workspace(rows, n_head, n_kv_head, head_dim, device="cuda"):
    """The (zeroed once, reusable) workspace ullm_hip_qkv_proj_append needs for
    this shape, or None; cached per shape and device."""
    n = _proj_ws_bytes(rows, n_head, n_kv_head, head_dim)
    if n == 0:
        return None
    key = (str(device), rows, n_head, n_kv_head, head_dim)
    ws = _proj_ws.get(key)
    if ws is None:
        ws = _proj_ws[key] = torch.zeros(n, dtype=torch.uint8, device=device)
    return ws


def _gemm_pays(rows, n, in_dim, head_dim, w_dtype):
    """Whether `rows` token rows of an [n, in_dim] projection run faster as
    ullm_hip_qkv_gemm_append (every weight read once, three launches) than as
    qkv_proj_append's matvec per row.  Measured (us, matvec / GEMM, 24 bits):
    16-bit weights: bf16 2560 -> 6144: 8 rows 20 / 20, 12 rows 29 / 20, 300 rows
    509 / 48; f16 2048 -> 3072: 24 rows 22 / 17; bf16 8192 -> 10240: 2 rows 62 /
    46; one row never gains (16384 -> 18432 122 / 152, f16 122 / 170).
    f32 weights are split into planes on each call, which a few rows do not pay
    for however large they are: 2560 -> 6144 16 rows 56 / 58, 24 rows 86 / 59;
    4096 -> 6144 16 rows 86 / 96, 20 rows 109 / 97; 8192 -> 10240 8 rows 235 /
    294, 12 rows 302 / 293; 16384 -> 18432 2 rows 365 / 1165, 12 rows 1529 / 1176.
    head_dim 256 from 256 head vectors on, where the matvec is 4 to 9 times
    slower (3584 -> 8192 6 / 8 rows: bf16 37 / 223 against 26, f32 62 / 203
    against 91); f32 8192 -> 32768: 2 rows 508 / 912, 3 rows 940 / 919; f32 512 ->
    8192: 8 rows (one round of 256 workgroups) 27 / 30, 9 rows 45 / 30."""
    f32 = w_dtype == torch.float32
    heads = rows * (n // head_dim)
    if head_dim == 256 and heads >= 256 and not (f32 and (rows < 3 or (heads == 256 and in_dim < 768))):
        return True
    work = rows * n * in_dim
    if f32:
        return (rows >= 20 and work >= 320_000_000) or (rows >= 12 and work >= 800_000_000)
    return rows > 1 and work >= 160_000_000


def qkv_proj_append(x, w_q, w_k, w_v, k_cache, v_cache, rope_cs, *, start_pos, n_head,
                    n_kv_head, head_dim, rotary_dim=None, neox=True, q_norm=None, k_norm=None,
                    eps=1e-6, q_bias=None, k_bias=None, v_bias=None, q_out=None, q_dtype=None,
                    kv_stride=None, workspace=None, stream=None):
    """Q/K/V projection (matvec_q, math.rs:9-21) with the append fused in
    (lib.rs:857-914).  x: [rows, in_dim] f32; w_*: [out, in_dim] f32/f16/bf16.
    Returns q_out ([rows, n_head*D], q_dtype); K/V land in the cache.  Few rows
    run as a matvec per row, whose workspace defaults to a cached one per shape
    (one caller at a time, as for GpuForward); more rows (`_gemm_pays`) as one
    GEMM with scratch of its own (rows x outputs x 4 bytes per range of in_dim,
    and x in planes: ullm_hip_qkv_gemm_workspace_bytes), `workspace` unused, or
    row by row where that memory is not there."""
    rows, in_dim = x.shape
    n = (n_head + 2 * n_kv_head) * head_dim
    args = (x, w_q, w_k, w_v, k_cache, v_cache, start_pos)
    prep = (rope_cs, n_head, n_kv_head, head_dim, rotary_dim, neox, q_norm, k_norm, eps, q_bias, k_bias,
            v_bias, q_out, q_dtype, kv_stride)
    if rows <= 65535 and _gemm_pays(rows, n, in_dim, head_dim, w_q.dtype):
        q = _F.proj(*args, 24, *prep, None, stream)
        if q is not None:
            return q
    if workspace is None:
        workspace = proj_workspace(rows, n_head, n_kv_head, head_dim, x.device)
    return _F.proj(*args, 0, *prep, workspace, stream)


def matmul(w, x, y=None, *, stream=None):
    """Batched projection y = x . w^T (forward.rs:675-726, shader.metal:519-566).
    w: [out, in] bf16; x: [n_cols, in] f32; y: [n_cols, out] f32 (allocated if
    None, else written in place, e.g. a view into an f32 KV cache)."""
    _need_cuda(w, x)
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1]:
        raise L.UllmHipError(L.E_INVALID, f"shapes w {tuple(w.shape)} x {tuple(x.shape)}")
    if x.dtype != torch.float32 or not x.is_contiguous() or not w.is_contiguous():
        raise L.UllmHipError(L.E_INVALID, "x must be contiguous f32 and w contiguous")
    n_cols, in_dim = x.shape
    out_dim = w.shape[0]
    if y is None:
        y = torch.empty(n_cols, out_dim, dtype=torch.float32, device=x.device)
    elif y.dtype != torch.float32 or tuple(y.shape) != (n_cols, out_dim) or not y.is_contiguous():
        raise L.UllmHipError(L.E_INVALID, "y must be contiguous f32 [n_cols, out]")
    L.check(L.lib().ullm_hip_matmul(_ptr(w), _dt(w), _ptr(x), _ptr(y), in_dim, out_dim, n_cols,
                                    _stream(stream)))
    return y


@dataclass
class AttnParams:
    """The attention fields of the reference's GpuParams (forward.rs:23-51)."""

    n_layer: int
    n_head: int
    n_kv_head: int
    head_dim: int
    n_ctx: int
    rope_theta: float = 10000.0
    eps: float = 1e-6
    rope_neox: bool = True
    rotary_dim: Optional[int] = None
    sliding_window: int = 0
    kv_dtype: torch.dtype = torch.float16


class GpuAttention:
    """Resident KV cache + the attention ops of one model, on one GPU.

    Mirrors what `GpuForward` owns and does for attention: the cache is
    `[n_layer][n_ctx][n_kv_head*head_dim]` (forward.rs:355-356), per-token
    decode appends then attends (forward.rs:414-466), batched prefill
    appends all rows then runs one causal attention (forward.rs:799-858),
    and Gemma-style local layers (`l % 6 != 5`) use the sliding window
    (forward.rs:450-454, :857).  Like GpuForward it is not thread-safe:
    one caller at a time (forward.rs:221-225).
    """

    def __init__(self, p: AttnParams, device="cuda"):
        if p.n_head % p.n_kv_head:
            raise L.UllmHipError(L.E_INVALID, "n_head must be a multiple of n_kv_head")
        self.p = p
        self.device = torch.device(device)
        self.rotary_dim = p.rotary_dim or p.head_dim
        self.kv_dim = p.n_kv_head * p.head_dim
        self.scale = 1.0 / math.sqrt(p.head_dim)
        shape = (p.n_layer, p.n_ctx, self.kv_dim)
        self.key_cache = torch.zeros(shape, dtype=p.kv_dtype, device=self.device)
        self.val_cache = torch.zeros(shape, dtype=p.kv_dtype, device=self.device)
        self.rope_cs = rope_table(p.n_ctx, self.rotary_dim, p.rope_theta, device=self.device)
        self.workspace = new_decode_workspace(1, p.n_head, p.n_kv_head, p.head_dim, p.n_ctx,
                                              0, self.device)
        # seq_lens for every position, uploaded once: decoding at pos passes
        # the device slice holding pos + 1 (no per-token copy or fill, nothing
        # for a captured graph to replay but kernels).
        self._lens = torch.arange(1, p.n_ctx + 1, dtype=torch.int32, device=self.device)

    def supports_batched_prefill(self) -> bool:
        """Prefill runs on MFMA for every cache dtype and head_dim (an f32
        cache with Q.K on bf16 hi + lo halves)."""
        return True

    def _window(self, layer: int) -> int:
        p = self.p
        return p.sliding_window if (p.sliding_window > 0 and layer % 6 != 5) else 0

    def _append(self, layer, q, k, v, start_pos, q_dtype, norms, biases):
        p = self.p
        qn, kn = norms
        qb, kb, vb = biases
        return qkv_append(q, k, v, self.key_cache[layer], self.val_cache[layer], self.rope_cs,
                          start_pos=start_pos, n_head=p.n_head, n_kv_head=p.n_kv_head,
                          head_dim=p.head_dim, rotary_dim=self.rotary_dim, neox=p.rope_neox,
                          q_norm=qn, k_norm=kn, eps=p.eps, q_bias=qb, k_bias=kb, v_bias=vb,
                          q_dtype=q_dtype)

    def _project_append(self, layer, xbs, wq, wk, wv, start_pos, norms, biases):
        """The prompt's bf16 projections and append: a few rows as matvecs (f32
        sums), more as one GEMM over the three weights (16 significant bits of
        xbs, as ullm_hip_matmul).  None where the operands are not what those
        take.  2560 -> 6144, us: 8 rows 21 (matvec), 40 rows 21, 2048 rows 129,
        against 87, 89 and 171 of three matmuls and the append."""
        p = self.p
        D, n = p.head_dim, (p.n_head + 2 * p.n_kv_head) * p.head_dim
        if not (xbs.is_cuda and xbs.dim() == 2 and xbs.dtype == torch.float32 and xbs.is_contiguous()
                and xbs.shape[0] > 0 and xbs.shape[1] >= 8 and xbs.shape[1] % 8 == 0
                and xbs.data_ptr() % 16 == 0):
            return None
        for w, m in ((wq, p.n_head), (wk, p.n_kv_head), (wv, p.n_kv_head)):
            if not (w.is_cuda and w.dtype == torch.bfloat16 and tuple(w.shape) == (m * D, xbs.shape[1])
                    and w.is_contiguous() and w.data_ptr() % 16 == 0):
                return None
        rows = xbs.shape[0]
        kc, vc = self.key_cache[layer], self.val_cache[layer]
        if rows < 32 and not _gemm_pays(rows, n, xbs.shape[1], D, wq.dtype):
            # Counters and partial rows of this call alone: prompts of several
            # engines, on several streams or threads, share nothing here.
            nb = _proj_ws_bytes(rows, p.n_head, p.n_kv_head, D)
            ws = torch.zeros(nb, dtype=torch.uint8, device=xbs.device) if nb else None
            return qkv_proj_append(xbs, wq, wk, wv, kc, vc, self.rope_cs, start_pos=start_pos,
                                   n_head=p.n_head, n_kv_head=p.n_kv_head, head_dim=D,
                                   rotary_dim=self.rotary_dim, neox=p.rope_neox, q_norm=norms[0],
                                   k_norm=norms[1], eps=p.eps, q_bias=biases[0],
                                   k_bias=biases[1], v_bias=biases[2], q_dtype=p.kv_dtype,
                                   workspace=ws)
        return _F.proj(xbs, wq, wk, wv, kc, vc, start_pos, 16, self.rope_cs, p.n_head, p.n_kv_head, D,
                       self.rotary_dim, p.rope_neox, norms[0], norms[1], p.eps, *biases, None,
                       p.kv_dtype, None, None, None)

    def forward(self, layer: int, q, k, v, pos: int, q_norm=None, k_norm=None, q_bias=None,
                k_bias=None, v_bias=None):
        """Decode one token: q [n_head*D], k/v [n_kv_head*D] f32 projections.
        Returns the attention output [n_head*D] f32."""
        p = self.p
        if not 0 <= pos < p.n_ctx:
            raise L.UllmHipError(L.E_INVALID, f"pos {pos} outside the context")
        return self._token(False, layer, pos, q_norm, k_norm, q_bias, k_bias, v_bias, q, k, v, None,
                           None)

    def _token(self, proj, layer, pos, q_norm, k_norm, q_bias, k_bias, v_bias, *ins):
        """Append or projection (proj), then attention, of one token in one
        native call; `ins`: q, k, v or the hidden state, the weights and the
        projection's workspace."""
        p = self.p
        return _F.token(proj, layer, pos, self.key_cache, self.val_cache, self._lens, self.workspace,
                        self._window(layer), self.scale, self.rope_cs, p.n_head, p.n_kv_head,
                        p.head_dim, self.rotary_dim, p.rope_neox, q_norm, k_norm, p.eps, q_bias,
                        k_bias, v_bias, *ins)

    def forward_batch(self, layer: int, q, k, v, start_pos: int = 0, q_norm=None, k_norm=None,
                      q_bias=None, k_bias=None, v_bias=None):
        """Prefill S tokens at start_pos..: q [S, n_head*D], k/v [S, kv_dim] f32.
        Returns the attention output [S, n_head*D] f32."""
        p = self.p
        S = q.shape[0]
        if start_pos + S > p.n_ctx:
            raise L.UllmHipError(L.E_INVALID, "prompt exceeds the context")
        qr = self._append(layer, q, k, v, start_pos, p.kv_dtype, (q_norm, k_norm),
                          (q_bias, k_bias, v_bias))
        return attn_prefill(qr, self.key_cache[layer], self.val_cache[layer], p.n_head,
                            p.n_kv_head, p.head_dim, start_pos=start_pos,
                            window=self._window(layer), scale=self.scale)

    # ---- attention blocks from the normed hidden state ----

    def forward_proj(self, layer: int, xb, pos: int, wq, wk, wv, q_norm=None, k_norm=None,
                     q_bias=None, k_bias=None, v_bias=None):
        """Decode one token from the attention-normed hidden state xb [n_embd]
        f32 (forward.rs:415-466): the Q/K/V matvecs in one launch, then the
        attention's two launches, which prepare q and the token's key (bias,
        norm, RoPE) and store its cache row.  Where those do not take the shape
        (the first 33 positions, head_dim 256, partial rotary, unaligned rows):
        the projection with the append fused in, then decode attention."""
        p = self.p
        if not 0 <= pos < p.n_ctx:
            raise L.UllmHipError(L.E_INVALID, f"pos {pos} outside the context")
        return self._token(True, layer, pos, q_norm, k_norm, q_bias, k_bias, v_bias, xb, wq, wk, wv,
                           proj_workspace(1, p.n_head, p.n_kv_head, p.head_dim, xb.device))

    def forward_batch_proj(self, layer: int, xbs, wq, wk, wv, start_pos: int = 0, q_norm=None,
                           k_norm=None, q_bias=None, k_bias=None, v_bias=None):
        """Prefill S tokens from the attention-normed hidden states xbs
        [S, n_embd] f32 (forward.rs:799-858): the three projections
        (forward.rs:799-801) as one MFMA GEMM with the append behind it, for few
        rows as a matvec per row (`_gemm_pays`), then causal prefill attention.
        bf16 weights take 16 significant bits of xbs, other weight dtypes 22 or
        24 (ullm_hip_qkv_gemm_append)."""
        p = self.p
        S = xbs.shape[0]
        if start_pos + S > p.n_ctx:
            raise L.UllmHipError(L.E_INVALID, "prompt exceeds the context")
        if wq.dtype == torch.bfloat16:
            qr = self._project_append(layer, xbs, wq, wk, wv, start_pos, (q_norm, k_norm),
                                      (q_bias, k_bias, v_bias))
            if qr is not None:
                return attn_prefill(qr, self.key_cache[layer], self.val_cache[layer], p.n_head,
                                    p.n_kv_head, p.head_dim, start_pos=start_pos,
                                    window=self._window(layer), scale=self.scale)
            q = matmul(wq, xbs)
            k = matmul(wk, xbs)
            v = matmul(wv, xbs)
            return self.forward_batch(layer, q, k, v, start_pos, q_norm, k_norm, q_bias, k_bias,
                                      v_bias)
        q_dtype = torch.float32 if p.kv_dtype == torch.float32 else p.kv_dtype
        qr = qkv_proj_append(xbs, wq, wk, wv, self.key_cache[layer], self.val_cache[layer],
                             self.rope_cs, start_pos=start_pos, n_head=p.n_head,
                             n_kv_head=p.n_kv_head, head_dim=p.head_dim,
                             rotary_dim=self.rotary_dim, neox=p.rope_neox, q_norm=q_norm,
                             k_norm=k_norm, eps=p.eps, q_bias=q_bias, k_bias=k_bias,
                             v_bias=v_bias, q_dtype=q_dtype)
        return attn_prefill(qr, self.key_cache[layer], self.val_cache[layer], p.n_head,
                            p.n_kv_head, p.head_dim, start_pos=start_pos,
                            window=self._window(layer), scale=self.scale)


    # ---- numerical debugging ----

    def forward_debug(self, xb, pos: int, wq, wk, wv, q_norm=None, k_norm=None, q_bias=None,
                      k_bias=None, v_bias=None, layer: int = 0, log=True):
        """The attention half of GpuForward::forward_debug (forward.rs:530-635):
        layer 0's attention one op at a time from the normed hidden state xb,
        each op its own launch followed by a synchronisation, reporting the
        NaN count, inf count and largest finite |value| of every intermediate
        (printed as `[dbg posP] label nan=.. inf=.. maxabs=..` when `log`, as
        the reference prints them).  The fused kernels are run with their
        later stages switched off to expose the intermediates: the raw
        projections come from the fused projection at position 0 with no
        norm or bias (RoPE at position 0 is the identity), then the bias,
        the Q/K norms and RoPE follow as appends into scratch rows, and the
        last append writes the cache row as forward_proj does (which sums the
        projections in another order: equal to f32 rounding).  The
        attention scores are never materialised by this path, so the report
        goes from rope_k to attn_out.  Returns (attention output, report:
        a list of (label, nan, inf, maxabs))."""
        p = self.p
        if not 0 <= pos < p.n_ctx:
            raise L.UllmHipError(L.E_INVALID, f"pos {pos} outside the context")
        report = []

        def check(t, label):
            torch.cuda.synchronize()
            v = t.detach().float().reshape(-1).cpu()
            nan = int(torch.isnan(v).sum())
            inf = int(torch.isinf(v).sum())
            fin = v[torch.isfinite(v)]
            mx = float(fin.abs().max()) if fin.numel() else 0.0
            report.append((label, nan, inf, mx))
            if log:
                import sys

                print(f"[dbg pos{pos}] {label:<14} nan={nan} inf={inf} maxabs={mx:.4f}",
                      file=sys.stderr)

        dev, kd = self.device, self.kv_dim
        x = xb.view(1, -1)
        check(x, "attn_in")
        # raw projections: scratch f32 K/V row 0, identity RoPE, no norm/bias
        sk = torch.zeros(1, kd, device=dev)
        sv = torch.zeros_like(sk)
        q_raw = qkv_proj_append(x, wq, wk, wv, sk, sv, self.rope_cs, start_pos=0,
                                n_head=p.n_head, n_kv_head=p.n_kv_head, head_dim=p.head_dim,
                                rotary_dim=self.rotary_dim, neox=p.rope_neox,
                                q_dtype=torch.float32)
        k_raw, v_raw = sk.clone(), sv.clone()
        check(q_raw, "wq")
        check(k_raw, "wk")
        check(v_raw, "wv")

        def scratch_append(norms, biases, at):
            ck = torch.zeros(at + 1, kd, device=dev)
            cv = torch.zeros_like(ck)
            qo = qkv_append(q_raw, k_raw, v_raw, ck, cv, self.rope_cs, start_pos=at,
                            n_head=p.n_head, n_kv_head=p.n_kv_head, head_dim=p.head_dim,
                            rotary_dim=self.rotary_dim, neox=p.rope_neox, q_norm=norms[0],
                            k_norm=norms[1], eps=p.eps, q_bias=biases[0], k_bias=biases[1],
                            v_bias=biases[2], q_dtype=torch.float32)
            return qo, ck[at], cv[at]

        biases = (q_bias, k_bias, v_bias)
        if any(b is not None for b in biases):
            qb_, kb_, vb_ = scratch_append((None, None), biases, 0)
            check(qb_, "bias_q")
            check(kb_, "bias_k")
            check(vb_, "bias_v")
        if q_norm is not None or k_norm is not None:
            qn_, kn_, _ = scratch_append((q_norm, k_norm), biases, 0)
            if q_norm is not None:
                check(qn_, "q_norm")
            if k_norm is not None:
                check(kn_, "k_norm")
        # the real append: RoPE at pos, K/V into the cache (as forward_proj)
        qr = self._append(layer, q_raw, k_raw, v_raw, pos, torch.float32, (q_norm, k_norm),
                          biases)
        check(qr, "rope_q")
        check(self.key_cache[layer, pos], "rope_k")
        out = attn_decode(qr.view(1, p.n_head, p.head_dim), self.key_cache[layer],
                          self.val_cache[layer], self._lens[pos:pos + 1], pos + 1, p.n_kv_head,
                          window=self._window(layer), scale=self.scale,
                          workspace=self.workspace)
        check(out, "attn_out")
        return out.view(-1), report
