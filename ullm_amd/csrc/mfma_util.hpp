// Device helpers shared by the MFMA attention kernels: 16-bit packing, MFMA
// wrappers, buffer resources, LDS DMA and LDS reads that bypass the
// compiler's LDS-DMA alias tracking.
#pragma once
#include "common.hpp"

namespace ullm {

constexpr int kRsrcWord3 = 0x00020000;  // raw buffer resource word 3 (gfx9 data format)

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Pointer known to be wave-uniform, kept in SGPRs.
__device__ __forceinline__ void *uniform_ptr(const void *p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (void *)(((uint64_t)hi << 32) | lo);
}

// Compile-time loop: f(Int<0>{}) ... f(Int<N-1>{}).
template <int V>
struct Int { static constexpr int value = V; };
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(Int<I>{});
        static_for<I + 1, N>(f);
    }
}

// Compiler-only ordering point for wave-private LDS traffic.
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

template <class T>
__device__ __forceinline__ f32x4 mfma16(const u32x4 &a, const u32x4 &b, const f32x4 &c) {
    if constexpr (__is_same(T, BF16))
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// Pair of f32 -> packed 16-bit pair of T (hardware RNE), and back.
template <class T>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (__is_same(T, BF16)) return pack_bf16x2(a, b);
    else return pack_f16x2(a, b);
}
template <class T>
__device__ __forceinline__ void unpack2(uint32_t w, float &a, float &b) {
    if constexpr (__is_same(T, BF16)) { a = bf16_lo(w); b = bf16_hi(w); }
    else { a = f16_lo(w); b = f16_hi(w); }
}
// x = hi + lo with hi, lo in T: ~2x the mantissa bits of T.
// Returns {hi, lo} packed pairs.
template <class T>
__device__ __forceinline__ u32x2 split2(float x0, float x1) {
    const uint32_t hi = pack2<T>(x0, x1);
    float h0, h1;
    unpack2<T>(hi, h0, h1);
    return u32x2{hi, pack2<T>(x0 - h0, x1 - h1)};
}

// s_waitcnt immediate that waits until at most n vector-memory operations
// are outstanding (gfx9 encoding: vmcnt[3:0] | vmcnt[5:4] << 14; expcnt and
// lgkmcnt left at their maxima).
constexpr int vm_wait(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }


typedef __attribute__((address_space(3))) void lds_void;

// LDS reads of DMA-filled tiles, issued as inline asm: the compiler would
// otherwise treat every LDS read as possibly aliasing in-flight LDS DMA and
// wait for all of it (vmcnt(0)), serialising the two-stage pipeline.  The
// caller waits with lds_wait() (tied to the destination registers) before use.
// One 16-byte-per-lane buffer load straight into LDS (lane i -> dst + 16 i),
// nontemporal.  Offsets past the resource's range read zero; the range check
// covers the per-lane offset, so callers put every variable part there and
// keep the scalar offset at 0.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, char *dst, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 16, voff, soff, 0, 2);
}
// Same load with the default cache policy, for operands that other
// workgroups re-read from L2 (GEMM tiles).
__device__ __forceinline__ void dma16_cached(__amdgpu_buffer_rsrc_t r, char *dst, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)p;
}
__device__ __forceinline__ u32x4 lds_read_b128(uint32_t a) {
    u32x4 r;
    asm volatile("ds_read_b128 %0, %1" : "=v"(r) : "v"(a));
    return r;
}
__device__ __forceinline__ void lds_write_b128(uint32_t a, const u32x4 &v) {
    asm volatile("ds_write_b128 %0, %1" ::"v"(a), "v"(v) : "memory");
}
__device__ __forceinline__ void lds_write_b64(uint32_t a, const u32x2 &v) {
    asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(v) : "memory");
}
__device__ __forceinline__ u32x2 lds_read_tr16_b64(uint32_t a) {
    u32x2 r;
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(r) : "v"(a));
    return r;
}
// 16-byte-per-lane raw buffer load that the compiler does not track: it
// would otherwise make every later use wait for all vector-memory traffic
// issued after it (vmcnt retires in order, LDS DMA included).  The caller
// waits with an explicit vmcnt wait and ties the registers before use.  The
// resource is a raw descriptor {base lo, base hi, bytes, word3} in SGPRs.
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i32x4 raw_rsrc(const void *base, int bytes) {
    const uint64_t v = (uint64_t)base;
    return i32x4{(int)__builtin_amdgcn_readfirstlane((uint32_t)v),
                 (int)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32) & 0xffff),
                 __builtin_amdgcn_readfirstlane(bytes), kRsrcWord3};
}
__device__ __forceinline__ u32x4 buffer_load_b128_untracked(const i32x4 &rsrc, int voff) {
    u32x4 v;
    asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen" : "=v"(v) : "v"(voff), "s"(rsrc) : "memory");
    return v;
}

// Same reads with a compile-time byte offset in the instruction's immediate
// field (0..65535), so per-lane addresses can be computed once.
template <int OFF>
__device__ __forceinline__ u32x4 lds_read_b128_at(uint32_t a) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset");
    u32x4 r;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(a), "i"(OFF));
    return r;
}
template <int OFF>
__device__ __forceinline__ u32x2 lds_read_tr16_b64_at(uint32_t a) {
    static_assert(OFF >= 0 && OFF < 65536, "ds offset");
    u32x2 r;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(a), "i"(OFF));
    return r;
}
// Waits until at most N LDS reads of this wave are outstanding (they retire
// in order, so the earlier ones are complete).
template <int N>
__device__ __forceinline__ void lds_wait_n() {
    static_assert(N >= 0 && N < 16, "lgkmcnt");
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(N) : "memory");
}
// max(x[l], x[l ^ 32]) across the wave halves, without an LDS round trip.
__device__ __forceinline__ float max_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <int N>
__device__ __forceinline__ void lds_wait(u32x4 (&r)[N]) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("" : "+v"(r[i]));
}

}  // namespace ullm

namespace ullm {

template <class T>
__device__ __forceinline__ f32x16 mfma32(const u32x4 &a, const u32x4 &b, const f32x16 &c) {
    if constexpr (__is_same(T, BF16))
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// Waits for this wave's outstanding LDS reads and ties the results to the
// wait so the compiler cannot use them earlier.
__device__ __forceinline__ void lds_wait_any() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void tie(u32x4 &r) { asm volatile("" : "+v"(r)); }
__device__ __forceinline__ void tie_f(float &r) { asm volatile("" : "+v"(r)); }
// One 4-byte LDS read per lane, not tracked by the compiler (see the 16-byte
// reads above); the caller waits with lds_wait_any() and ties the result.
__device__ __forceinline__ uint32_t lds_read_b32(uint32_t a) {
    uint32_t r;
    asm volatile("ds_read_b32 %0, %1" : "=v"(r) : "v"(a));
    return r;
}
__device__ __forceinline__ void tie(u32x2 &r) { asm volatile("" : "+v"(r)); }

// Workgroup barrier without a memory fence (LDS DMA visibility is ensured by
// each wave's own vmcnt wait before it).
__device__ __forceinline__ void wg_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Paged K/V (tab == nullptr: the contiguous cache).  Key t of the sequence
// is row t % P of page tab[t / P] (P = 2^shift, a multiple of every prefill
// kernel's key tile), so a tile's DMA goes through a buffer resource based at its page
// whose range ends at the sequence length: rows past it, and pages outside
// the table or [0, n_pages), read as zeros.
struct KvPages {
    const int32_t *tab;
    int tab_len, shift, n_pages;
};

// Buffer resources and scalar offset of the key tile starting at key0 (a
// tile never crosses a page).  EB: bytes per cache element.
template <int D, int EB = 2>
__device__ __forceinline__ void page_tile(const KvPages &pg, const char *kc, const char *vc,
                                          int kvh, int rbg, int kv_len, int key0,
                                          __amdgpu_buffer_rsrc_t &kr, __amdgpu_buffer_rsrc_t &vr,
                                          int &so) {
    const int pi = key0 >> pg.shift;
    const int phys = key0 < kv_len && pi < pg.tab_len ? pg.tab[pi] : -1;
    const bool ok = phys >= 0 && phys < pg.n_pages;
    const int64_t pb = ((int64_t)(ok ? phys : 0) << pg.shift) * rbg + (int64_t)kvh * D * EB;
    const int rows = min(1 << pg.shift, kv_len - (pi << pg.shift));
    const int range = ok ? (rows - 1) * rbg + D * EB : 0;
    kr = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(kc + pb), 0, range, kRsrcWord3);
    vr = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(vc + pb), 0, range, kRsrcWord3);
    so = __builtin_amdgcn_readfirstlane((key0 & ((1 << pg.shift) - 1)) * rbg);
}

// Prefill with the key ranges split over workgroups.  The query rows are taken
// in units of UR rows and the keys in tiles of `tile`; a unit of more than
// `chunk` tiles is cut into parts of equal tile counts, each a workgroup of its
// own that leaves (m, l) and the unnormalised O of its rows, which
// launch_prefill_merge adds up.  Part p's O is a whole [S][n_head*D] plane,
// its (m, l) a [S][n_head] plane of pairs.  No unit has more than the `parts`
// parts that are launched and have planes.
struct KeySplit {
    int chunk, parts, tile;
    float *o;
    float2 *ml;
};
// Key tiles [t0, t1) of unit u: the window start of its first row to the
// causal end of its last.
__host__ __device__ __forceinline__ void unit_tiles(int u, int UR, int S, int start_pos, int window,
                                                    int tile, int &t0, int &t1) {
    const int hi = start_pos + (u * UR + UR < S ? u * UR + UR : S);
    const int lo = window > 0 && start_pos + u * UR + 1 - window > 0 ? start_pos + u * UR + 1 - window : 0;
    t0 = lo / tile;
    t1 = (hi + tile - 1) / tile;
}
// Parts of a unit of n tiles.
__device__ __forceinline__ int unit_parts(const KeySplit &sp, int n) {
    return min((n + sp.chunk - 1) / sp.chunk, sp.parts);
}
// The unit's parts, and part `part`'s share of [t0, t1).
__device__ __forceinline__ int part_tiles(const KeySplit &sp, int part, int &t0, int &t1) {
    const int parts = unit_parts(sp, t1 - t0), per = (t1 - t0 + parts - 1) / parts;
    t0 += part * per;
    t1 = min(t1, t0 + per);
    return parts;
}
int launch_prefill_merge(int D, KeySplit sp, int UR, int S, int start_pos, int window, int n_head,
                         float *out, hipStream_t st);
// Host: the split of a call.  chunk: tiles per part of the longest unit, which
// has `parts` of them; bytes: the scratch for O and (m, l).  kUncut: one part
// for a unit of any length, and no scratch.
struct SplitPlan {
    int chunk, parts;
    size_t ml_off, bytes;
};
constexpr SplitPlan kUncut{0x3fffffff, 1, 0, 0};
// The units of a call: n workgroups' worth of them when unsplit (row units
// times head groups), the longest and the average one in key tiles.
struct UnitLoad {
    double n, longest, avg;
};
// Unit lengths never fall from one whole unit to the next (they grow with the
// causal end until the window's start leaves key 0; from there UR, a multiple
// of `tile` wherever a window is given, moves both ends by whole tiles), so the
// longest is the last unit or, when S cuts that one short, the one before it.
// (Units of half a tile are only estimated with: to within a tile.)
inline UnitLoad unit_load(int S, int UR, int n_hg, int start_pos, int window, int tile) {
    const int n = (S + UR - 1) / UR;
    auto len = [&](int u, int &t0) {
        int t1;
        unit_tiles(u, UR, S, start_pos, window, tile, t0, t1);
        return t1 - t0;
    };
    int a0, b0, p0;
    const int first = len(0, a0), last = len(n - 1, b0), prev = len(n > 1 ? n - 2 : 0, p0);
    const int longest = last > prev ? last : prev;
    // lengths grow to a window's size, and stay there
    const bool flat = window > 0 && b0 > 0;
    const double ramp = flat && window > start_pos ? (double)(window - start_pos) / S : 0.;
    const double avg = flat ? longest - ramp * 0.5 * (longest - first) : 0.5 * (first + last);
    return UnitLoad{(double)n * n_hg, (double)longest, avg};
}
// What a workgroup of a prefill kernel costs (us): per key tile when it has
// the chip nearly alone and when every CU runs one, and once per workgroup.
struct PrefillCost {
    double alone, full, fixed;
};
// Estimated time of `wgs` workgroups over `total` tiles, the longest of
// `longest` (one workgroup per CU at a time).
inline double prefill_us(const PrefillCost &c, double wgs, double longest, double total) {
    const double fill = wgs < 256 ? wgs / 256 : 1., ts = c.alone + (c.full - c.alone) * fill;
    const int rounds = (int)((wgs + 255) / 256);
    // equal workgroups run in whole rounds; unequal ones fill each other's gaps
    const double avg = total / wgs, even = longest * rounds, mixed = total / 256 + 0.5 * avg;
    const double tiles = avg > 0.9 * longest ? even : (mixed > longest ? mixed : longest);
    return tiles * ts + c.fixed * rounds;
}
// The number of parts with the least estimate, against `unsplit` us without a
// split (0: one part on the same kernel); the merge streams the partial results
// at 4 TB/s.  A split has to win by an eighth and by 1.5 us: timed over 146
// random shapes (2..4096 rows at 0..16384, all dtypes and head_dims) the calls
// that it splits ran 1.1 to 13 times faster, and none of the others moved.
inline SplitPlan choose_split(const PrefillCost &c, const UnitLoad &u, double unsplit, int S, int n_head,
                              int D) {
    static const int env = env_override("ULLM_HIP_PREFILL_PARTS");  // tuning: parts of the longest unit (1: never)
    SplitPlan pl = kUncut;
    if (!(unsplit > 0)) unsplit = prefill_us(c, u.n, u.longest, u.n * u.avg);
    double best = unsplit * 0.875 < unsplit - 1.5 ? unsplit * 0.875 : unsplit - 1.5;
    if (u.n > 1024 && env < 2) return pl;  // the chip is full many times over
    for (int p : {2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 40, 48, 64}) {
        if (env > 0 ? p != env : 2 * p > u.longest + 1) continue;
        const int chunk = ((int)u.longest + p - 1) / p, parts = ((int)u.longest + chunk - 1) / chunk;
        const size_t ml_off = (size_t)parts * S * n_head * D * 4;
        if (parts < 2 || ml_off > (256u << 20)) continue;
        double mean = u.avg > 0.9 * u.longest ? parts : u.avg / chunk + 0.5;
        mean = mean > parts ? parts : (mean < 1 ? 1 : mean);
        const double us = prefill_us(c, u.n * mean, chunk, u.n * u.avg) + 2.5 +
                          (double)S * n_head * D * 4 * (2 * mean + 1) / 4e6;
        if (us < best || env > 1) {
            best = us;
            pl = SplitPlan{chunk, parts, ml_off, ml_off + (size_t)parts * S * n_head * 8};
        }
    }
    return pl;
}
inline KeySplit split_at(const SplitPlan &pl, int tile, void *ws) {
    return KeySplit{pl.chunk, pl.parts, tile, (float *)ws, (float2 *)((char *)ws + pl.ml_off)};
}

// Head_dim-256 prefill on 16-row waves, two per SIMD (prefill16.hip);
// pgs.tab == nullptr for a contiguous cache.
// ws: scratch for a split of the key ranges over workgroups, used where the
// plan asks for one and ws_bytes holds it (ullm_hip_prefill_workspace_bytes).
int launch_prefill16(int dtype, const void *q, const void *kc, const void *vc, int64_t kvs, int S,
                     int start_pos, int window, int n_head, int kv_mul, float qs, float *out,
                     hipStream_t st, KvPages pgs, void *ws = nullptr, size_t ws_bytes = 0);
// The split prefill16_kernel takes for these shapes, and the estimate (us) of
// the call without one.
SplitPlan prefill16_split(int dtype, int S, int start_pos, int window, int n_head, int kv_mul, int D);
double prefill16_us(int dtype, int S, int start_pos, int window, int n_head, int kv_mul, int D);
int launch_prefill16_128(int dtype, const void *q, const void *kc, const void *vc, int64_t kvs,
                         int S, int start_pos, int window, int n_head, int kv_mul, float qs,
                         float *out, hipStream_t st, KvPages pgs, void *ws = nullptr,
                         size_t ws_bytes = 0);

}  // namespace ullm
