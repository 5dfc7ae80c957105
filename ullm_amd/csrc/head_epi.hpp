// One head vector per wave: bias/norm/RoPE epilogue of the decode projection
// and of the decode step's merge, and typed loads and stores.
#pragma once
#include "common.hpp"
#include "wave.hpp"

namespace ullm {

template <int E>
__device__ __forceinline__ void load_e(const float *p, float (&x)[E]) {
    if constexpr (E == 1) x[0] = p[0];
    else if constexpr (E == 2) { const float2 v = *(const float2 *)p; x[0] = v.x; x[1] = v.y; }
    else { const float4 v = *(const float4 *)p; x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w; }
}

// Store E consecutive elements converted to OUT_DT.
template <int OUT_DT, int E>
__device__ __forceinline__ void store_e(void *base, int64_t idx, const float (&x)[E]) {
    if constexpr (OUT_DT == ULLM_DT_F32) {
        float *p = (float *)base + idx;
        if constexpr (E == 1) p[0] = x[0];
        else if constexpr (E == 2) *(float2 *)p = float2{x[0], x[1]};
        else *(float4 *)p = float4{x[0], x[1], x[2], x[3]};
    } else {
        // hardware round-to-nearest-even packs
        auto pk = [](float a, float b) {
            return OUT_DT == ULLM_DT_F16 ? pack_f16x2(a, b) : pack_bf16x2(a, b);
        };
        uint16_t *p = (uint16_t *)base + idx;
        if constexpr (E == 1) p[0] = (uint16_t)pk(x[0], 0.f);
        else if constexpr (E == 2) *(uint32_t *)p = pk(x[0], x[1]);
        else *(uint2 *)p = uint2{pk(x[0], x[1]), pk(x[2], x[3])};
    }
}

// Per-lane state of the head epilogue of one token row: the (cos, sin) of
// this lane's elements at the row's position and the Q/K norm weights.  A
// lane holds E = D/64 consecutive elements of a head vector.
template <int D>
struct HeadEpi {
    static constexpr int E = D / 64;
    int lane, e0, rotary_dim, half, neox;
    float eps;
    float rc[E], rs[E], wq[E], wk[E];
    const float *q_norm, *k_norm;

    __device__ __forceinline__ HeadEpi(const float *cs, int pos, int rotary_dim_, int neox_,
                                       const float *qn, const float *kn, float eps_)
        : lane((int)(threadIdx.x & 63)), e0((int)(threadIdx.x & 63) * E), rotary_dim(rotary_dim_),
          half(rotary_dim_ / 2), neox(neox_), eps(eps_), q_norm(qn), k_norm(kn) {
        const float *cp = cs + (int64_t)pos * half * 2;
#pragma unroll
        for (int i = 0; i < E; i++) {
            const int e = e0 + i;
            const int j = e < rotary_dim ? (neox ? (e < half ? e : e - half) : e >> 1) : 0;
            rc[i] = cp[2 * j];
            rs[i] = cp[2 * j + 1];
            wq[i] = 1.f;
            wk[i] = 1.f;
        }
        if (q_norm) load_e<E>(q_norm + e0, wq);
        if (k_norm) load_e<E>(k_norm + e0, wk);
    }

    // Bias (already added by the caller), per-head RMSNorm (math.rs:82-86)
    // and RoPE (math.rs:116-161) of one head vector of kind 0 (q), 1 (k) or
    // 2 (v), in the reference's order.  lds_row: D floats private to the
    // wave, used only for partial-rotary pairs.
    __device__ __forceinline__ void norm_rope(float (&x)[E], int kind, float *lds_row) const {
        const float *nw = kind == 0 ? q_norm : (kind == 1 ? k_norm : nullptr);
        if (nw) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < E; i++) ss += x[i] * x[i];
            ss = wave_sum(ss);
            // v_rsq_f32 (~1 ulp) for (sum/n + eps).sqrt().recip()
            const float inv = __builtin_amdgcn_rsqf(ss / (float)D + eps);
#pragma unroll
            for (int i = 0; i < E; i++) x[i] = x[i] * inv * (kind == 0 ? wq[i] : wk[i]);
        }
        if (kind == 2) return;
        float y[E];
        if (rotary_dim == D) {
            // Full-width RoPE: a NeoX partner (e +- D/2) sits in lane l ^ 32 at
            // the same element index; an interleaved partner (e ^ 1) in the same
            // lane, or in lane l ^ 1 when a lane holds one element.
#pragma unroll
            for (int i = 0; i < E; i++) {
                float pa;
                if (neox) pa = xor32(x[i]);
                else if constexpr (E == 1) pa = dpp<kDppXor1>(x[i]);
                else pa = x[i ^ 1];
                const bool lo = neox ? lane < 32 : ((e0 + i) & 1) == 0;
                // lo: a*c - b*s with a = own, b = partner; hi: a*s + b*c with a = partner
                y[i] = lo ? x[i] * rc[i] - pa * rs[i] : pa * rs[i] + x[i] * rc[i];
            }
        } else {
            // Partial rotary: the partner of each pair comes from the wave's
            // LDS row (LDS operations of one wave complete in order).
#pragma unroll
            for (int i = 0; i < E; i++) lds_row[e0 + i] = x[i];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < E; i++) {
                const int e = e0 + i;
                y[i] = x[i];
                if (e < rotary_dim) {
                    if (neox) {
                        const int j = e < half ? e : e - half;
                        const float a = lds_row[j], c = lds_row[j + half];
                        y[i] = e < half ? a * rc[i] - c * rs[i] : a * rs[i] + c * rc[i];
                    } else {
                        const float a = lds_row[e & ~1], c = lds_row[e | 1];
                        y[i] = (e & 1) ? a * rs[i] + c * rc[i] : a * rc[i] - c * rs[i];
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();  // the row may be rewritten next
        }
#pragma unroll
        for (int i = 0; i < E; i++) x[i] = y[i];
    }
};

}  // namespace ullm
