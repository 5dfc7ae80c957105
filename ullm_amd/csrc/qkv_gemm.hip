// Q/K/V projection of many token rows as one MFMA GEMM over the three weight
// matrices, feeding the fused append: what qkv_proj_append computes
// (crates/ullm-model/src/lib.rs:857-914 per token, the batched form of the
// reference's forward.rs:799-853) without re-reading the weights per row.
//
//   split_rows_kernel   X (f32)  -> NP 16-bit planes whose sum is X
//   qkv_gemm_kernel     Y[ks] = X . [W_q; W_k; W_v]^T over one key range each
//   qkv_append_kernel   sum over ks, bias, norm, RoPE, q and cache rows
//
// Planes.  The matrix cores take 16-bit operands, their products are exact
// and they add in f32, so the precision is that of the planes:
//   bf16 weights: X = 2 bf16 planes (16 significant bits, what
//     ullm_hip_matmul carries) or 3 (24 bits: every f32 exactly);
//   f16 weights: X scaled by a power of two per row (its largest finite |x|
//     in [2^14, 2^15)) into 2 f16 planes, the second times 2^12: 22 bits (at
//     least: what f16 leaves of a value is rounded to f16 again), and never less
//     than 2^-51 of the row's largest value; each plane has its own sum, and the
//     scales are taken out of those and of Y;
//   f32 weights: X and W as 3 bf16 planes each, the six products of weight
//     2^-16 and above.
//
// qkv_gemm_kernel.  8 waves in two sets of four, one wave of each set on
// every SIMD, half a step apart: while one set runs the MFMAs of its step
// from registers, the other reads its next step's fragments from LDS and
// issues DMA, and they swap at a workgroup barrier.  Tiles go global -> LDS
// by buffer loads into a ring of NST stages of 32 KU input dims.
#include <algorithm>
#include "common.hpp"
#include "mfma_util.hpp"
#include "wave.hpp"

namespace ullm {

constexpr int kGmK = 32;                // input dims of one row of a tile
constexpr int kGmRB = kGmK * 2;         // its bytes
constexpr int kGmPad = 128;             // X and W planes: dims padded to a multiple (zeros)
constexpr int kGmOOB = 0x7ffffff0;      // buffer offset past every valid range: reads zero
constexpr float kLowPlane = 0x1p-12f;   // scale of the second f16 plane

struct GemmArgs {
    const char *wq, *wk, *wv;  // [n_q][in_dim] ...; NW > 1: wq = the planes [NW][n][ldx]
    const char *xp;            // X planes [NP][rows][ldx]
    const float *inv;          // per-row factor of Y, or nullptr
    float *y;                  // [ks][rows][n]
    int n_q, n_kv, n;          // outputs: q, k (and v), all
    int in_dim, ldx, rows;     // ldx: in_dim padded
    int mt, nt, ks;            // tiles of tokens and outputs, key ranges
    const float *x;            // the operands themselves: [rows][in_dim],
    const char *w[3];          // W_q, W_k, W_v
};

// SI x OI blocks of 32 x 32 per wave, WS x WO waves, NP planes of X and NW of
// W, KU x 32 dims per step.
template <int NW, int NP, int SI, int OI, int WS, int WO, int KU, int NST>
struct GemmCfg {
    static_assert(WS * WO == 8, "8 waves");
    static constexpr int BS = 32 * SI * WS, BO = 32 * OI * WO;
    static constexpr int WROWS = NW * BO, XROWS = NP * BS;    // 64-byte rows per 32 dims
    static constexpr int NI = (WROWS + XROWS) / 16;           // 1 KiB DMA instructions per 32 dims
    static constexpr int NDMA = (NI * KU + 7) / 8;            // ... per step and wave
    static constexpr int STAGE = NDMA * 8 * 1024;
    static_assert(NST * STAGE <= 160 * 1024, "LDS");
};

// 16-byte slot swizzle of a 64-byte row: 4 rows share a 256-byte bank line.
__device__ __forceinline__ int gm_swz(int r) { return (r >> 2) & 3; }

// Output o of token row s over input dims [d0, d1), in f32: NaN as soon as the sum is.
template <class T, int NW>
__device__ float plain_dot(const GemmArgs &a, int s, int o, int d0, int d1) {
    const int m = o < a.n_q ? 0 : (o < a.n_q + a.n_kv ? 1 : 2);
    const int64_t row = o - (m == 0 ? 0 : (m == 1 ? a.n_q : a.n_q + a.n_kv));
    const float *xr = a.x + (int64_t)s * a.in_dim;
    float sum = 0.f;
    for (int d = d0; d < d1 && sum == sum; d += 4) {
        const float4 v = *(const float4 *)(xr + d);
        float w[4];
        if constexpr (NW == 3) {
            const float4 t = *(const float4 *)((const float *)a.w[m] + row * a.in_dim + d);
            w[0] = t.x, w[1] = t.y, w[2] = t.z, w[3] = t.w;
        } else {
            const uint2 t = *(const uint2 *)((const uint16_t *)a.w[m] + row * a.in_dim + d);
            unpack2<T>(t.x, w[0], w[1]);
            unpack2<T>(t.y, w[2], w[3]);
        }
        sum = __builtin_fmaf(w[0], v.x, sum);
        sum = __builtin_fmaf(w[1], v.y, sum);
        sum = __builtin_fmaf(w[2], v.z, sum);
        sum = __builtin_fmaf(w[3], v.w, sum);
    }
    return sum;
}

template <class T, int NW, int NP, int SI, int OI, int WS, int WO, int KU, int NST, bool FOLD>
__global__ __launch_bounds__(512) void qkv_gemm_kernel(GemmArgs a) {
    using C = GemmCfg<NW, NP, SI, OI, WS, WO, KU, NST>;
    constexpr int BS = C::BS, BO = C::BO, STAGE = C::STAGE, NDMA = C::NDMA;
    constexpr int KD = KU * kGmK, SUB = C::NI * 1024;  // dims per step, LDS bytes per 32 dims
    __shared__ __attribute__((aligned(1024))) char lds[NST * STAGE];

    // Workgroup i runs on XCD i % 8; each XCD takes a contiguous run of tiles,
    // token tile fastest, so the tiles it holds share W rows in its L2.
    const int total = a.mt * a.nt * a.ks;
    const int per_xcd = (total + 7) / 8;
    const int t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (t >= total) return;
    const int s0 = (t % a.mt) * BS, o0 = (t / a.mt) % a.nt * BO, part = t / (a.mt * a.nt);
    const int nk = (a.in_dim + KD - 1) / KD;
    const int kb = (int)((int64_t)nk * part / a.ks), ke = (int)((int64_t)nk * (part + 1) / a.ks);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int set = wave >> 2;

    // DMA plan: a stage is, for each 32 dims, WROWS rows of W planes, then
    // XROWS of X planes; 16 rows per instruction, instructions NDMA wave .. + NDMA - 1 by this
    // wave.  Lane i fills slot i % 4 of row i / 4, holding chunk slot ^ swz.
    // The matrix of an instruction's W rows is wave-uniform: the boundaries
    // between W_q, W_k and W_v are multiples of 64 rows.
    __amdgpu_buffer_rsrc_t rs[NDMA];
    int dofs[NDMA];
    bool cut[NDMA];  // chunk past in_dim in the last step
    const int tail = a.in_dim - (nk - 1) * KD;
#pragma unroll
    for (int c = 0; c < NDMA; c++) {
        const int ins = wave * NDMA + c, u = ins / C::NI;  // wave-uniform
        const int r0 = (ins - u * C::NI) * 16, r = r0 + lane / 4;
        const int dk = u * kGmK + ((lane & 3) ^ gm_swz(r)) * 8;
        const char *base;
        int range, row, rows, ld;
        cut[c] = false;
        if (u < KU && r0 < C::WROWS) {
            const int ob = o0 + r0 % BO;
            if constexpr (NW == 1) {
                const bool isq = ob < a.n_q, isk = !isq && ob < a.n_q + a.n_kv;
                base = isq ? a.wq : (isk ? a.wk : a.wv);
                row = ob - (isq ? 0 : (isk ? a.n_q : a.n_q + a.n_kv)) + lane / 4;
                rows = isq ? a.n_q : a.n_kv;
                ld = a.in_dim;
                cut[c] = dk >= tail;
            } else {
                base = a.wq + (int64_t)(r0 / BO) * a.n * a.ldx * 2;
                row = ob + lane / 4;
                rows = a.n;
                ld = a.ldx;
            }
        } else {
            const int x0 = r0 - C::WROWS;
            base = a.xp + (int64_t)(x0 / BS) * a.rows * a.ldx * 2;
            row = s0 + x0 % BS + lane / 4;
            rows = u < KU ? a.rows : 0;
            ld = a.ldx;
        }
        range = (int)((int64_t)rows * ld * 2);
        rs[c] = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(base), 0, __builtin_amdgcn_readfirstlane(range), kRsrcWord3);
        dofs[c] = row < rows ? (row * ld + dk) * 2 : kGmOOB;
    }
    // Loads of step k into its stage; steps past the end re-read the last one
    // (never used), so every step issues the same count.
    auto issue = [&](int k) {
        char *dst = lds + ((k - kb) % NST) * STAGE + wave * NDMA * 1024;
        const int kk = min(k, ke - 1);
        const bool last = kk == nk - 1;
#pragma unroll
        for (int c = 0; c < NDMA; c++)
            dma16_cached(rs[c], dst + c * 1024, last && cut[c] ? kGmOOB : dofs[c], kk * KD * 2);
    };

    // Per-lane fragment addresses in stage 0: row c32 of a 32-row block, the
    // 8 dims of half h2 of each k16 step.  Blocks are 32 rows apart and share
    // the swizzle, so block, plane and stage are added as constants.
    const int c32 = lane & 31, h2 = lane >> 5;
    const int wm = wave % WS, wn = wave / WS;
    const uint32_t lds0 = lds_addr(lds);
    uint32_t aw[2], ax[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t slot = ((2 * h + h2) ^ gm_swz(c32)) * 16;
        aw[h] = lds0 + (wn * 32 * OI + c32) * kGmRB + slot;
        ax[h] = lds0 + (C::WROWS + wm * 32 * SI + c32) * kGmRB + slot;
    }

    // FOLD: the matrix cores sum one step from zero, smallest products first,
    // into acc[0] and acc[1] in turn (BYP: each plane of X into its own).  The
    // step before is added to `sum` in f32 in the shadow of the MFMAs, and every
    // eight steps `sum` goes to `top`, so that few additions round at the size of
    // the whole result.  Relative error at in_dim 2048..2560 (f64 reference):
    // 0.9e-7..1.1e-7, against 1.2e-7..1.3e-7 of qkv_proj_kernel's f32 sums and
    // 2.5e-7..5.6e-7 of one chain of MFMAs.
    constexpr bool BYP = FOLD && __is_same(T, F16);
    constexpr int NA = FOLD ? 2 : 1;
    f32x16 acc[NA][OI][SI], sum[FOLD ? OI : 1][FOLD ? SI : 1], top[FOLD ? OI : 1][FOLD ? SI : 1];
#pragma unroll
    for (int i = 0; i < OI; i++)
#pragma unroll
        for (int j = 0; j < SI; j++) {
#pragma unroll
            for (int n = 0; n < NA; n++) acc[n][i][j] = f32x16{};
            if constexpr (FOLD) sum[i][j] = top[i][j] = f32x16{};
        }
    auto raise = [&](int k) {
        if constexpr (FOLD)
            if (((k - kb) & 7) == 0) {
#pragma unroll
                for (int i = 0; i < OI; i++)
#pragma unroll
                    for (int j = 0; j < SI; j++) {
                        top[i][j] += sum[i][j];
                        sum[i][j] = f32x16{};
                    }
            }
    };

    u32x4 fw[2 * KU][NW][OI], fx[2 * KU][NP][SI];
    auto read = [&](int k) {
        const uint32_t so = ((k - kb) % NST) * STAGE;
        static_for<0, 2 * KU>([&](auto hc) {
            constexpr int h = decltype(hc)::value, U = h / 2 * SUB;
            const uint32_t w0 = aw[h & 1] + so, x0 = ax[h & 1] + so;
            static_for<0, NW * OI>([&](auto ic) {
                constexpr int p = decltype(ic)::value / OI, i = decltype(ic)::value % OI;
                fw[h][p][i] = lds_read_b128_at<U + (p * BO + i * 32) * kGmRB>(w0);
            });
            static_for<0, NP * SI>([&](auto ic) {
                constexpr int p = decltype(ic)::value / SI, i = decltype(ic)::value % SI;
                fx[h][p][i] = lds_read_b128_at<U + (p * BS + i * 32) * kGmRB>(x0);
            });
        });
    };
    auto landed = [&] {  // this wave's fragments are in their registers
        lds_wait_any();
#pragma unroll
        for (int h = 0; h < 2 * KU; h++) {
#pragma unroll
            for (int p = 0; p < NW; p++)
#pragma unroll
                for (int i = 0; i < OI; i++) tie(fw[h][p][i]);
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int i = 0; i < SI; i++) tie(fx[h][p][i]);
        }
    };
    constexpr int NMF = 2 * KU * OI * SI * (NW == 3 ? 6 : NP);  // MFMAs per step
    // BYP: plane 1 of this step while plane 0 of the step before is added to
    // `sum`, then plane 0 while plane 1 is added (twice the additions, under the
    // same MFMAs: 1000 rows x 2048 -> 3072 38.6 -> 39.0 us, traced).
    auto by_plane = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        constexpr int NM = 2 * KU * OI * SI, V = (OI * SI * 16 + NM - 1) / NM + 1;
        static_for<0, 2 * KU>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
#pragma unroll
            for (int i = 0; i < OI; i++)
#pragma unroll
                for (int j = 0; j < SI; j++)
                    acc[p][i][j] = mfma32<T>(fw[h][0][i], fx[h][p][j], h == 0 ? f32x16{} : acc[p][i][j]);
        });
#pragma unroll
        for (int i = 0; i < OI; i++)
#pragma unroll
            for (int j = 0; j < SI; j++) {
                if constexpr (p == 1) sum[i][j] += acc[0][i][j];
                else sum[i][j] += acc[1][i][j] * kLowPlane;
            }
        static_for<0, NM>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
        });
    };
    auto multiply = [&](auto nc) {
        constexpr int n = decltype(nc)::value;
        __builtin_amdgcn_s_setprio(1);
        if constexpr (BYP) {
            by_plane(Int<1>{});
            by_plane(Int<0>{});
            __builtin_amdgcn_s_setprio(0);
            return;
        }
        // products of plane weight 2, 1, 0 (FOLD), or plane by plane
        static_for<0, FOLD ? 3 : 1>([&](auto oc) {
            constexpr int ord = 2 - decltype(oc)::value;
            static_for<0, 2 * KU * NW * NP>([&](auto pc) {
                constexpr int h = decltype(pc)::value / (NW * NP);
                constexpr int pw = decltype(pc)::value / NP % NW, px = decltype(pc)::value % NP;
                if constexpr (!FOLD || pw + px == ord) {
                    constexpr bool lead = FOLD && h == 0 && pw == 0 && px == NP - 1;  // the first
#pragma unroll
                    for (int i = 0; i < OI; i++)
#pragma unroll
                        for (int j = 0; j < SI; j++)
                            acc[n][i][j] = mfma32<T>(fw[h][pw][i], fx[h][px][j],
                                                     lead ? f32x16{} : acc[n][i][j]);
                }
            });
        });
        if constexpr (FOLD) {
#pragma unroll
            for (int i = 0; i < OI; i++)
#pragma unroll
                for (int j = 0; j < SI; j++) sum[i][j] += acc[1 - n][i][j];
            constexpr int V = (OI * SI * 16 + NMF - 1) / NMF + 1;
            static_for<0, NMF>([&](auto) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, V, 0);  // V additions
            });
        }
        __builtin_amdgcn_s_setprio(0);
    };
    auto meet = [&] {
        __builtin_amdgcn_sched_barrier(0);
        wg_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // Own DMA of the step after the newest NST - 2 issued has landed.
    auto dma_wait = [&] { __builtin_amdgcn_s_waitcnt(vm_wait((NST - 2) * NDMA)); };

    // Phases p = 0, 1, ..., a barrier after each.  Set 0 reads step kb + i in
    // phase 2i and multiplies in 2i + 1; set 1 reads it in 2i + 1 and
    // multiplies in 2i + 2.  Step i's stage is last read in phase 2i + 1, so
    // from phase 2i + 2 on it is refilled with step i + NST; every wave has
    // waited for its share of step i + 1 by the end of phase 2i + 1.
#pragma unroll
    for (int i = 0; i < NST - 1; i++) issue(kb + i);
    dma_wait();
    meet();
    auto turn = [&](auto setc, auto nc, int k) {
        constexpr int SET = decltype(setc)::value;
        read(k);
        issue(k + NST - 1);
        raise(k);
        landed();
        if (SET == 1) dma_wait();
        meet();
        multiply(nc);
        if (SET == 0) dma_wait();
        meet();
    };
    auto run = [&](auto setc) {
        for (int k = kb; k < ke; k += NA) {
            turn(setc, Int<0>{}, k);
            if (NA == 2 && k + 1 < ke) turn(setc, Int<NA - 1>{}, k + 1);
        }
    };
    if (set == 0) {
        run(Int<0>{});
        meet();
    } else {
        meet();
        run(Int<1>{});
    }
    __builtin_amdgcn_s_waitcnt(vm_wait(0));  // the unused loads past the end

    // acc[i][j][4 g + e] = Y[s, o]: s = s0 + (wm SI + j) 32 + c32,
    // o = o0 + (wn OI + i) 32 + 8 g + 4 h2 + e.
    if constexpr (FOLD) {  // the last step's sums are not added yet
        const bool odd = BYP || ((ke - kb) & 1);
#pragma unroll
        for (int i = 0; i < OI; i++)
#pragma unroll
            for (int j = 0; j < SI; j++) {
                const f32x16 even = top[i][j] + (sum[i][j] + acc[0][i][j]);
                const f32x16 other = top[i][j] + (sum[i][j] + acc[NA - 1][i][j]);
#pragma unroll
                for (int e = 0; e < 16; e++) acc[0][i][j][e] = odd ? even[e] : other[e];
            }
    }
    float *yp = a.y + (int64_t)part * a.rows * a.n;
    bool nan = false;
#pragma unroll
    for (int j = 0; j < SI; j++) {
        const int s = s0 + (wm * SI + j) * 32 + c32;
        if (s >= a.rows) continue;
        const float f = a.inv ? a.inv[s] : 1.f;
        float *yr = yp + (int64_t)s * a.n;
#pragma unroll
        for (int i = 0; i < OI; i++) {
            const int ob = o0 + (wn * OI + i) * 32 + 4 * h2;
#pragma unroll
            for (int g = 0; g < 4; g++)
                if (ob + 8 * g < a.n) {
                    const f32x4 v = f32x4{acc[0][i][j][4 * g] * f, acc[0][i][j][4 * g + 1] * f,
                                          acc[0][i][j][4 * g + 2] * f, acc[0][i][j][4 * g + 3] * f};
                    *(f32x4 *)(yr + ob + 8 * g) = v;
                    if constexpr (FOLD) nan |= v[0] != v[0] || v[1] != v[1] || v[2] != v[2] || v[3] != v[3];
                }
        }
    }
    // An infinite weight times a plane of x that is zero, or of the other sign,
    // makes NaN of what is an infinity: outputs that are NaN are summed again
    // from the operands (rarely any; a real NaN ends its sum where it is met).
    if constexpr (FOLD)
        if (nan) {
            const int d0 = kb * KD, d1 = min(ke * KD, a.in_dim);
#pragma unroll 1
            for (int b = 0; b < SI * OI * 16; b++) {
                const int j = b / (OI * 16), i = b / 16 % OI;
                const int s = s0 + (wm * SI + j) * 32 + c32;
                const int o = o0 + (wn * OI + i) * 32 + 4 * h2 + (b % 16 / 4) * 8 + b % 4;
                if (s >= a.rows || o >= a.n) continue;
                float *yo = yp + (int64_t)s * a.n + o;
                if (*yo != *yo) *yo = plain_dot<T, NW>(a, s, o, d0, d1);
            }
        }
}

// x = the sum of NP values of T.  An infinity or NaN goes to the last plane
// alone (it meets the other operand's first plane only, so an infinity times
// a finite value stays one), and a finite x whose rounding to T would
// overflow takes T's largest value first.
template <class T, int NP>
__device__ __forceinline__ void planes_of(float x, uint16_t (&o)[NP]) {
    constexpr float kBig = __is_same(T, BF16) ? 0x1.fep127f : 65504.f;
    const bool fin = __builtin_fabsf(x) < __builtin_inff();
    float r = fin ? x : 0.f;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const uint32_t h = pack2<T>(fminf(fmaxf(r, -kBig), kBig), 0.f) & 0xffffu;
        o[p] = (uint16_t)h;
        float hf, z;
        unpack2<T>(h, hf, z);
        r -= hf;
        // |r| <= half a step of a value below 2^15 (2^3): 2^15 at most
        if constexpr (__is_same(T, F16)) r *= 1.f / kLowPlane;
    }
    if (!fin) o[NP - 1] = (uint16_t)(pack2<T>(x, 0.f) & 0xffffu);
}

// Rows of f32 into NP planes of T, [NP][rows][ld] (dims past in_dim zero),
// one row per workgroup.  SCALE: the row is multiplied by the power of two
// that puts its largest finite |x| in [2^14, 2^15) first, inv[row] undoing it.
// Streams 4 + 2 NP bytes per element; the SCALE row's second pass hits L1/L2.
template <class T, int NP, bool SCALE>
__global__ __launch_bounds__(256) void split_rows_kernel(const float *__restrict__ x0,
                                                         const float *__restrict__ x1,
                                                         const float *__restrict__ x2, int r1, int r2,
                                                         int in_dim, int ld, int rows,
                                                         uint16_t *__restrict__ out,
                                                         float *__restrict__ inv) {
    const int row = blockIdx.x;
    const float *xr = (row < r1 ? x0 + (int64_t)row * in_dim
                                : (row < r2 ? x1 + (int64_t)(row - r1) * in_dim
                                            : x2 + (int64_t)(row - r2) * in_dim));
    float f = 1.f;
    if constexpr (SCALE) {
        __shared__ float wmax[4];
        float m = 0.f;
        for (int i = threadIdx.x * 4; i < in_dim; i += 1024) {
            const float4 v = *(const float4 *)(xr + i);
            const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float b = __builtin_fabsf(e[c]);
                m = b < __builtin_inff() ? fmaxf(m, b) : m;
            }
        }
        m = wave_max(m);
        if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
        __syncthreads();
        m = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
        // biased exponent of m; the scale 2^(14 - e) and its inverse both stay normal
        const int e = max((int)(__float_as_uint(m) >> 23), 16) - 127;
        f = m > 0.f ? __uint_as_float((uint32_t)(14 - e + 127) << 23) : 1.f;
        if (threadIdx.x == 0) inv[row] = m > 0.f ? __uint_as_float((uint32_t)(e - 14 + 127) << 23) : 1.f;
    }
    for (int i = threadIdx.x * 8; i < ld; i += 2048) {
        float e[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (i < in_dim) {  // in_dim is a multiple of 8
            const float4 v0 = *(const float4 *)(xr + i), v1 = *(const float4 *)(xr + i + 4);
            e[0] = v0.x, e[1] = v0.y, e[2] = v0.z, e[3] = v0.w;
            e[4] = v1.x, e[5] = v1.y, e[6] = v1.z, e[7] = v1.w;
        }
        uint32_t w[NP][4];
#pragma unroll
        for (int c = 0; c < 8; c += 2) {
            uint16_t p0[NP], p1[NP];
            planes_of<T, NP>(e[c] * f, p0);
            planes_of<T, NP>(e[c + 1] * f, p1);
#pragma unroll
            for (int p = 0; p < NP; p++) w[p][c / 2] = p0[p] | ((uint32_t)p1[p] << 16);
        }
#pragma unroll
        for (int p = 0; p < NP; p++)
            *(u32x4 *)(out + ((int64_t)p * rows + row) * ld + i) = u32x4{w[p][0], w[p][1], w[p][2], w[p][3]};
    }
}

// ---- plan -------------------------------------------------------------------

enum GemmTile { kT128x384, kT128x256, kT128x128, kT64x256, kT64x128, kT32x256, kTiles };
// Tokens, outputs, and the share of the large tile's MFMA rate that the tile
// reaches (small tiles read more LDS bytes per product: measured with f16
// weights, 1000 rows x 2048 -> 3072, 0.49 us of MFMAs per 64 dims and tile of
// 128 x 128: 128 x 128 and 64 x 256 0.62 us, half of it 64 x 128 0.43, 32 x 256 0.46).
struct GemmTileInfo { int bs, bo; double rate; };
constexpr GemmTileInfo kGmTile[kTiles] = {{128, 384, 1.}, {128, 256, .9}, {128, 128, .8}, {64, 256, .8}, {64, 128, .58}, {32, 256, .54}};

struct GemmPlan {
    int tile, mt, nt, ks, np, nw;
    size_t x_off, inv_off, w_off, y_off, bytes;
};

// Tile and number of key ranges: the least of an estimate over the choices.  A
// round of 256 workgroups costs its 32-dim steps, the slowest of the MFMAs
// (4.3 TFLOP/s per CU in the large tile), the stage's bytes (90 GB/s per CU)
// and the barriers (0.2 us), plus 3 us of pipeline fill and stores; a split
// adds its partial sums' traffic (written, and read by the append).
// Qwen3-4B shape, 2560 -> 6144 bf16, whole call (split, GEMM, append), us:
//   2048 rows: 128 x 384 129 (256 tiles: one round; the GEMM 105, 1.23
//     PFLOP/s executed), 128 x 256 158, 128 x 128 179; the three
//     ullm_hip_matmul launches and the append it replaces: 171;
//   61 rows: 64 x 128 in 5 ranges (taken) 22.1, 4 ranges 21.8, 2 ranges 25.2, unsplit
//     35.9, 32 x 256 23.3; replaced: 90.
static bool gemm_plan(int rows, int in_dim, int w_dtype, int x_bits, int n, GemmPlan &pl) {
    const int ld = (in_dim + kGmPad - 1) / kGmPad * kGmPad, nk = ld / kGmK;
    pl.nw = w_dtype == ULLM_DT_F32 ? 3 : 1;
    pl.np = w_dtype == ULLM_DT_F32 || (w_dtype == ULLM_DT_BF16 && x_bits > 16) ? 3 : 2;
    const int prods = pl.nw == 3 ? 6 : pl.np;
    if ((int64_t)rows * ld * 2 > 0x7fff0000LL || (int64_t)n * ld * 2 > 0x7fff0000LL) return false;
    static const int env_t = env_override("ULLM_HIP_GEMM_TILE"), env_k = env_override("ULLM_HIP_GEMM_KS");  // tuning
    double best = 1e30;
    for (int t = 0; t < kTiles; t++) {
        const int bs = kGmTile[t].bs, bo = kGmTile[t].bo;
        if (pl.nw == 3 && bo > 128 && bs > 32) continue;  // W planes: the stages would not fit
        if (bs * bo > 128 * 128 && !(w_dtype == ULLM_DT_BF16 && pl.np == 2)) continue;  // registers (FOLD)
        if (env_t > 0 && t != env_t - 1) continue;
        const int mt = (rows + bs - 1) / bs, nt = (n + bo - 1) / bo;
        const double flop = 2.0 * bs * bo * kGmK * prods, stage = (pl.nw * bo + pl.np * bs) * (double)kGmRB;
        const double step = std::max(std::max(flop / (4.3e6 * kGmTile[t].rate), stage / 90e3), 0.2);  // us
        for (int ks = 1; ks <= std::min(16, nk / 8 > 1 ? nk / 8 : 1); ks++) {
            if (env_k > 0 && ks != env_k) continue;
            const int64_t wgs = (int64_t)mt * nt * ks;
            const double rounds = (double)((wgs + 255) / 256);
            const double us = rounds * (3.0 + step * ((nk + ks - 1) / ks)) +
                              (ks - 1) * (double)rows * n * 8 / 4e6;
            if (us < best) best = us, pl.tile = t, pl.mt = mt, pl.nt = nt, pl.ks = ks;
        }
    }
    if (best == 1e30) return false;
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    pl.x_off = 0;
    pl.inv_off = up((size_t)pl.np * rows * ld * 2);
    pl.w_off = pl.inv_off + up((size_t)rows * 4);
    pl.y_off = pl.w_off + (pl.nw == 3 ? up((size_t)3 * n * ld * 2) : 0);
    pl.bytes = pl.y_off + up((size_t)pl.ks * rows * n * 4);
    return true;
}

template <class T, int NW, int NP>
static void launch_gemm(int tile, const GemmArgs &a, hipStream_t st) {
    constexpr bool F = !(__is_same(T, BF16) && NP == 2);
    const int per_xcd = (a.mt * a.nt * a.ks + 7) / 8;
    const dim3 g((unsigned)per_xcd * 8), b(512);
    constexpr bool T3 = NP == 3;
#define GEMM(SI, OI, WS, WO, KU, NST) \
    launch_kernel((qkv_gemm_kernel<T, NW, NP, SI, OI, WS, WO, KU, NST, F>), g, b, 0, st, a)
    if constexpr (!F) {
        if (tile == kT128x384) { GEMM(2, 3, 2, 4, 1, 4); return; }
        if (tile == kT128x256) { GEMM(2, 2, 2, 4, 1, 4); return; }
    }
    if constexpr (NW == 1) {
        if (tile == kT64x256) { GEMM(1, 2, 2, 4, T3 ? 1 : 2, T3 ? 4 : 3); return; }
        if (tile == kT128x128) { GEMM(2, 1, 2, 4, T3 ? 1 : 2, T3 ? 4 : 3); return; }
        if (tile == kT64x128) { GEMM(1, 1, 2, 4, 2, T3 ? 3 : 4); return; }
        GEMM(1, 1, 1, 8, 2, T3 ? 3 : 4);
    } else {
        if (tile == kT128x128) { GEMM(2, 1, 2, 4, 1, 3); return; }
        if (tile == kT64x128) { GEMM(1, 1, 2, 4, 1, 4); return; }
        GEMM(1, 1, 1, 8, 1, 2);
    }
#undef GEMM
}

}  // namespace ullm

using namespace ullm;

static bool plan_call(int rows, int in_dim, int w_dtype, int x_bits, int n_head, int n_kv_head, int head_dim,
                      GemmPlan &pl) {
    return rows >= 1 && in_dim >= 8 && in_dim % 8 == 0 && dtype_ok(w_dtype) && (x_bits == 16 || x_bits == 24) &&
           n_head >= 1 && n_kv_head >= 1 && (head_dim == 64 || head_dim == 128 || head_dim == 256) &&
           ((int64_t)n_head + 2 * (int64_t)n_kv_head) * head_dim <= 0x7fffffff &&
           gemm_plan(rows, in_dim, w_dtype, x_bits, (n_head + 2 * n_kv_head) * head_dim, pl);
}

extern "C" size_t ullm_hip_qkv_gemm_workspace_bytes(int rows, int in_dim, int w_dtype, int x_bits,
                                                    int n_head, int n_kv_head, int head_dim) {
    GemmPlan pl;
    return plan_call(rows, in_dim, w_dtype, x_bits, n_head, n_kv_head, head_dim, pl) ? pl.bytes : 0;
}

extern "C" int ullm_hip_qkv_gemm_plan(int rows, int in_dim, int w_dtype, int x_bits, int n_head, int n_kv_head,
                                      int head_dim, int32_t *plan) {
    GemmPlan pl;
    if (!plan) return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_plan: null pointer");
    if (!plan_call(rows, in_dim, w_dtype, x_bits, n_head, n_kv_head, head_dim, pl))
        return set_error(ULLM_HIP_E_UNSUPPORTED, "qkv_gemm_plan: %d rows, %d -> %d/%d heads x %d, dtype %d", rows,
                         in_dim, n_head, n_kv_head, head_dim, w_dtype);
    plan[0] = kGmTile[pl.tile].bs, plan[1] = kGmTile[pl.tile].bo, plan[2] = pl.ks;
    return ULLM_HIP_OK;
}

extern "C" int ullm_hip_qkv_gemm_append(const float *x, int in_dim, const void *w_q,
                                        const void *w_k, const void *w_v, int w_dtype, int x_bits,
                                        const float *q_bias, const float *k_bias,
                                        const float *v_bias, const float *q_norm,
                                        const float *k_norm, float eps, const float *rope_cs,
                                        int rope_n_pos, int rope_neox, int rotary_dim, int rows,
                                        int start_pos, int n_head, int n_kv_head, int head_dim,
                                        void *q_out, int q_dtype, void *k_cache, void *v_cache,
                                        int kv_dtype, int64_t kv_stride, void *workspace,
                                        size_t workspace_bytes, void *stream) {
    if (!dtype_ok(w_dtype) || !dtype_ok(q_dtype) || !dtype_ok(kv_dtype))
        return set_error(ULLM_HIP_E_UNSUPPORTED, "qkv_gemm_append: dtype w=%d q=%d kv=%d", w_dtype,
                         q_dtype, kv_dtype);
    if (head_dim != 64 && head_dim != 128 && head_dim != 256)
        return set_error(ULLM_HIP_E_UNSUPPORTED, "qkv_gemm_append: head_dim %d not in {64,128,256}",
                         head_dim);
    if (x_bits != 16 && x_bits != 24)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: x_bits %d (16 or 24)", x_bits);
    if (rows < 0 || start_pos < 0 || n_head < 1 || n_kv_head < 1 || n_head % n_kv_head)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: bad rows/heads");
    if (in_dim < 8 || in_dim % 8)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: in_dim %d must be a positive multiple of 8",
                         in_dim);
    if (rotary_dim < 2 || rotary_dim > head_dim || (rotary_dim & 1))
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: rotary_dim %d", rotary_dim);
    if (kv_stride < (int64_t)n_kv_head * head_dim)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: kv_stride too small");
    if (rows == 0) return ULLM_HIP_OK;
    if (!x || !w_q || !w_k || !w_v || !rope_cs || !q_out || !k_cache || !v_cache)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: null tensor pointer");
    if (((uintptr_t)x | (uintptr_t)w_q | (uintptr_t)w_k | (uintptr_t)w_v) & 15)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: x and weights must be 16-byte aligned");
    if (rope_n_pos < (int64_t)start_pos + rows)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: rope table has %d positions, need %lld",
                         rope_n_pos, (long long)start_pos + rows);
    const int64_t n64 = ((int64_t)n_head + 2 * (int64_t)n_kv_head) * head_dim;
    GemmPlan pl;
    if (n64 > 0x7fffffff || !gemm_plan(rows, in_dim, w_dtype, x_bits, (int)n64, pl))
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: an operand of 2 GiB or more");
    if (!workspace || workspace_bytes < pl.bytes)
        return set_error(ULLM_HIP_E_WORKSPACE, "qkv_gemm_append: workspace of %zu bytes needed, %zu given",
                         pl.bytes, workspace_bytes);
    if ((uintptr_t)workspace & 255)
        return set_error(ULLM_HIP_E_INVALID, "qkv_gemm_append: workspace must be 256-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const int n = (int)n64, n_q = n_head * head_dim, n_kv = n_kv_head * head_dim;
    const int ld = (in_dim + kGmPad - 1) / kGmPad * kGmPad;
    char *ws = (char *)workspace;
    uint16_t *xp = (uint16_t *)(ws + pl.x_off);
    float *inv = (float *)(ws + pl.inv_off), *y = (float *)(ws + pl.y_off);
    const bool f16 = w_dtype == ULLM_DT_F16;
    GemmArgs a{(const char *)w_q, (const char *)w_k, (const char *)w_v, (const char *)xp,
               f16 ? inv : nullptr, y, n_q, n_kv, n, in_dim, ld, rows, pl.mt, pl.nt, pl.ks,
               x, {(const char *)w_q, (const char *)w_k, (const char *)w_v}};
    const dim3 xg((unsigned)rows), b(256);
    if (f16)
        launch_kernel((split_rows_kernel<F16, 2, true>), xg, b, 0, st, x, x, x, rows, rows, in_dim, ld, rows, xp, inv);
    else if (pl.np == 2)
        launch_kernel((split_rows_kernel<BF16, 2, false>), xg, b, 0, st, x, x, x, rows, rows, in_dim, ld, rows, xp, inv);
    else
        launch_kernel((split_rows_kernel<BF16, 3, false>), xg, b, 0, st, x, x, x, rows, rows, in_dim, ld, rows, xp, inv);
    if (pl.nw == 3) {
        uint16_t *wp = (uint16_t *)(ws + pl.w_off);
        launch_kernel((split_rows_kernel<BF16, 3, false>), dim3((unsigned)n), b, 0, st,
                           (const float *)w_q, (const float *)w_k, (const float *)w_v, n_q, n_q + n_kv,
                           in_dim, ld, n, wp, inv);
        a.wq = (const char *)wp;
        launch_gemm<BF16, 3, 3>(pl.tile, a, st);
    } else if (f16) {
        launch_gemm<F16, 1, 2>(pl.tile, a, st);
    } else if (pl.np == 2) {
        launch_gemm<BF16, 1, 2>(pl.tile, a, st);
    } else {
        launch_gemm<BF16, 1, 3>(pl.tile, a, st);
    }
    const int rc = check_hip(hipGetLastError(), "qkv_gemm launch");
    if (rc != ULLM_HIP_OK) return rc;
    return append_rows(y, y + n_q, y + n_q + n_kv, AppendSrc{n, n, pl.ks, (int64_t)rows * n}, q_bias, k_bias, v_bias,
                       q_norm, k_norm, eps, rope_cs, rope_neox, rotary_dim, rows, start_pos, n_head,
                       n_kv_head, head_dim, q_out, q_dtype, k_cache, v_cache, kv_dtype, kv_stride, st);
}
