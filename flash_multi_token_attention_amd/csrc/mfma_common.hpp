// Building blocks of the bf16 MFMA conv-attention kernels (gfx950, wave64).
//
// MFMA 16x16x32 register layout (lane = 16*g + n, g = 0..3, n = 0..15):
//   A operand: row n of the 16 x 32 tile, k = 8g .. 8g+7   (8 x 16-bit, one b128)
//   B operand: column n of the 32 x 16 tile, k = 8g .. 8g+7
//   C/D:       column n, rows 4g .. 4g+3                    (4 x fp32)
//
// The key-axis part of the (c_q x c_k) window is a banded Toeplitz matrix, so the
// convolution of a score tile is c_q MFMAs per 16 x 16 output block: for query
// tap a, C^T[16 out keys][16 queries] += T_a^T[16 x 32] * S^T[32 in keys][16
// queries shifted by a - pad_q rows].  The 32 input keys start 8 before the
// block's first output key (a 16-byte-aligned LDS column), which covers
// pad_k <= 8.  Scores are staged in LDS as fp16 (11-bit significand; bf16's 8
// bits would cost ~1e-2 in the softmax argument).
#pragma once
#include <atomic>
#include <type_traits>

#include "common.hpp"

namespace convattn {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x8 __attribute__((ext_vector_type(8)));
// Five consecutive dwords at a 4-byte boundary of LDS, as 32-bit reads (the compiler pairs them
// into ds_read2_b32).  A 128-bit LDS read that is not 16-byte aligned is legal on gfx950 but slow:
// measured with four waves reading, one costs about 66 clocks of the LDS pipe against about 12 for
// the five dwords read separately.
__device__ __forceinline__ void lds_read_dwords5(const unsigned char *p, u32x4 &lo, unsigned int &hi) {
    const unsigned int *q = reinterpret_cast<const unsigned int *>(p);
    lo = (u32x4){q[0], q[1], q[2], q[3]};
    hi = q[4];
}

constexpr int kKeyHalo = 8;          // LDS columns before a block's first output key
constexpr int kMfmaMaxPk = 8;        // so c_k <= 17 on the MFMA path
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kF16Max = 65504.f;   // what a score beyond fp16's range is rounded to

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_f16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// ---- The window of two query taps as one sparse matrix product ----
// v_smfmac_f32_16x16x64_f16 takes the issue time of the dense 16x16x32 (16.5 clocks per SIMD measured for both, one to four waves)
// and twice its k: of every four consecutive k of the B operand each row of A uses two, which two an index says.  A band of at
// most 15 keys fits that: of the keys kappa and kappa + 16 of a 32-key window an output key sees one at most.  With a dword (two
// keys) of the window's first 16-key block beside the same dword of its second, every group of four k is {kappa, kappa + 1,
// kappa + 16, kappa + 17}, and a row takes the first two or the last two.  Output key n sees the window's keys n + 1 .. n + 15,
// so it takes the first block's keys kappa, kappa + 1 where kappa + 1 > n and the second block's otherwise.
//
// B operand of lane (g, n): dwords 0..3 belong to the first tap, 4..7 to the second, each as {first block keys 4g, 4g+1; second
// block the same; first block keys 4g+2, 4g+3; second block}.  The two blocks may also stand the other way round, with the other index:
// a window that moves on by one block replaces the dwords of its older block only.
// A operand of lane (g, n): row n, the first tap for g < 2 and the second for the rest; its element 2q + e, q = 0..3, is key
// 4 (2 (g & 1) + q / 2) + 2 (q & 1) + e of the block the row takes; the index has 4 bits for each q.
__device__ __forceinline__ f32x4 smfmac_f16(f16x8 a, u32x8 b, f32x4 c, int index) {
    return __builtin_amdgcn_smfmac_f32_16x16x64_f16(a, __builtin_bit_cast(f16x16, b), c, index, 0, 0);
}
constexpr int kSparseMaxCk = 15;
__device__ __forceinline__ int sparse_key(int g, int q) { return 4 * (2 * (g & 1) + (q >> 1)) + 2 * (q & 1); }
// index of a lane where the window's first block has the even dwords (`swapped`: the odd ones)
__device__ __forceinline__ int sparse_index(int g, int n, bool swapped) {
    int v = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) v |= (((sparse_key(g, q) + 1 > n) != swapped) ? 0x4 : 0xE) << (4 * q);
    return v;
}
// Which taps share a product.  A window of CQT tap slots needs, for output rows of parity ob = 0 and 1, the score rows at
// offsets delta = slot - (CQT - 1) + ob, CQT + 1 of them.  Operand tuple j holds the offsets delta(j, 0) and delta(j, 1).  For an odd
// CQT the tuples hold all offsets in pairs, and one slot of each parity stays single: a dense product of four dwords of a tuple.  (Not
// a sparse one with zero weights for the other four: those are a row outside the window, whose infinities and NaN would get into the
// output row.  Nor the sparse 16x16x32: where the 16x16x64 one follows it on the same accumulators, the compiler's waits are too short.)
// For an even CQT they hold the offsets of parity 1, and parity 0 has, for its first and its last slot, a tuple of its own in the place
// of the last one.
template <int CQT> struct SparseTaps {
    static constexpr bool odd = CQT % 2 != 0;
    static constexpr int tuples = CQT / 2 + 1;   // operand tuples
    static constexpr int products = CQT / 2;     // sparse products per output parity
    static constexpr int delta(int j, int half) {
        return !odd && j == CQT / 2 ? (half ? 0 : -(CQT - 1)) : -(CQT - (odd ? 1 : 2)) + 2 * j + half;
    }
    // tuple of product i of parity ob
    static constexpr int tuple(int i, int ob) { return odd ? i + ob : !ob && i == CQT / 2 - 1 ? CQT / 2 : i; }
    // tap slot of a half of tuple j for parity ob
    static constexpr int slot(int j, int half, int ob) { return delta(j, half) + CQT - 1 - ob; }
    // the single slot of a parity (odd CQT): half ob of this tuple
    static constexpr int single_tuple(int ob) { return ob ? 0 : tuples - 1; }
    static constexpr int single_slot(int ob) { return slot(single_tuple(ob), ob, ob); }
    static constexpr bool every_slot_once() {
        for (int ob = 0; ob < 2; ++ob) {
            int seen = odd ? 1 << single_slot(ob) : 0;
            for (int x = 0; x < 2 * products; ++x) {
                const int t = slot(tuple(x / 2, ob), x % 2, ob);
                if (t < 0 || t >= CQT || (seen >> t & 1)) return false;
                seen |= 1 << t;
            }
            if (seen != (1 << CQT) - 1) return false;
        }
        return true;
    }
};
// The bands of a head as a table in LDS: dword x + 16 of tap slot t's 48 holds the weights of two neighbouring keys, T[x] and T[x + 1]
// with T[x] = w[a][pk + x - 8] * mul (zero outside the window), x = the key's place in the window less the output
// key's; slot t stands for tap a = t - (CQT - c_q).  A lane finds the pairs of its operands there with
// 4-byte reads: one or two loads of W per thread instead of the 48 to 88 gathers of every lane.
constexpr int kBandRow = 48;
template <int CQT> constexpr int band_table_bytes() { return CQT * kBandRow * 4; }
template <int CQT>
__device__ __forceinline__ void band_table_build(unsigned int *tab, const float *__restrict__ w_head, int c_q, int c_k, int pk, float mul,
                                                 int tid, int nthreads) {
    for (int i = tid; i < CQT * kBandRow; i += nthreads) {
        const int t = i / kBandRow, a = t - (CQT - c_q), off = i - t * kBandRow - 16 - kKeyHalo;
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int b = pk + off + e;
            v[e] = w_head[min(max(a, 0), c_q - 1) * c_k + min(max(b, 0), c_k - 1)];
            v[e] = a >= 0 && b >= 0 && b < c_k ? v[e] * mul : 0.f;
        }
        const f16x2 two = {(_Float16)v[0], (_Float16)v[1]};
        tab[i] = __builtin_bit_cast(unsigned int, two);
    }
}
// The A operands of both parities: band[ob][i] of product i, and of the single slot one[w][ob] where the window's first block has the
// even (w = 0) or, BOTH, the odd (w = 1) dwords.
template <int CQT, bool BOTH> struct SparseBands {
    using T = SparseTaps<CQT>;
    static_assert(T::every_slot_once(), "the slots of the products");
    f16x8 band[2][T::products], one[BOTH ? 2 : 1][2];
    // c + the single slot of parity ob, from the tuple it is in
    __device__ __forceinline__ f32x4 single(int w, int ob, u32x8 rows, f32x4 c) const {
        const u32x4 v = ob ? (u32x4){rows[4], rows[5], rows[6], rows[7]} : (u32x4){rows[0], rows[1], rows[2], rows[3]};
        if (!BOTH && w) return mfma_f16(one[0][ob], __builtin_bit_cast(f16x8, (u32x4){v[1], v[0], v[3], v[2]}), c);
        return mfma_f16(one[w][ob], __builtin_bit_cast(f16x8, v), c);
    }
    __device__ __forceinline__ void read(const unsigned int *tab, int g, int n) {
#pragma unroll
        for (int ob = 0; ob < 2; ++ob) {
#pragma unroll
            for (int i = 0; i < T::products; ++i) {
                const int j = T::tuple(i, ob);
                u32x4 v;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int kappa = sparse_key(g, q), x = kappa + (kappa + 1 > n ? 0 : 16) - n;
                    v[q] = tab[(g < 2 ? T::slot(j, 0, ob) : T::slot(j, 1, ob)) * kBandRow + x + 16];
                }
                band[ob][i] = __builtin_bit_cast(f16x8, v);
            }
            if constexpr (T::odd)
#pragma unroll
                for (int w = 0; w < (BOTH ? 2 : 1); ++w) {
                    u32x4 v;
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        v[q] = tab[T::single_slot(ob) * kBandRow + 4 * g + 2 * (q >> 1) + ((q & 1) != w ? 16 : 0) - n + 16];
                    one[w][ob] = __builtin_bit_cast(f16x8, v);
                }
        }
    }
};

// Scheduling hints: the sequence of these calls in program order is the order in which the
// backend lays out groups of LDS reads and MFMAs.  Used as "reads of stage s+1, then MFMAs
// of stage s" so that fragment reads stay one stage ahead instead of sinking next to their use.
#define SCHED_DS_READ(n) __builtin_amdgcn_sched_group_barrier(0x100, (n), 0)
#define SCHED_MFMA(n) __builtin_amdgcn_sched_group_barrier(0x008, (n), 0)
// The same with an explicit pipeline id: groups are only ordered against groups of their own id,
// and the backend places long pipelines badly, so every row block of a phase gets its own.
#define SCHED_DS_READ_ID(n, id) __builtin_amdgcn_sched_group_barrier(0x100, (n), (id))
#define SCHED_MFMA_ID(n, id) __builtin_amdgcn_sched_group_barrier(0x008, (n), (id))

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>): a loop whose index is a
// constant expression in the body (the scheduling-group builtins need one).
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Four raw scores to fp16, two per dword (one v_cvt_pkrtz_f16_f32 per pair).  Rounded toward zero:
// a finite score beyond fp16's range becomes +-65504 instead of infinity, so no clamp is needed.
// Every kernel of the forward and the backward rounds its scores with this function: P = exp2(C - LSE)
// only sums to one over a row if C is the C the forward's LSE was taken from.
__device__ __forceinline__ u32x2 pack_scores_f16(f32x4 s) {
    return (u32x2){__builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(s[0], s[1])),
                   __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(s[2], s[3]))};
}

// Bands for a compile-time tap count CQT >= c_q: the window is padded with zero
// taps in FRONT (older query rows), so tap slot t stands for tap a = t - (CQT - c_q)
// and reads score row  i + t - (CQT - 1); the padded slots read rows that exist
// (the halo above the tile) and multiply them by zero.  No run-time tap loop.
template <int CQT>
__device__ __forceinline__ void load_bands(f16x8 (&tf)[CQT], const float *__restrict__ w_head, int c_q,
                                           int c_k, int pk, int g, int n, bool flip, float mul) {
#pragma unroll
    for (int t = 0; t < CQT; ++t) {
        const int a = t - (CQT - c_q);
        f16x8 f = (f16x8)(_Float16)0.f;
        if (a >= 0) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                int b = 8 * g + e - kKeyHalo - n + pk;
                float v = 0.f;
                if (b >= 0 && b < c_k) v = w_head[a * c_k + (flip ? (c_k - 1 - b) : b)] * mul;
                f[e] = (_Float16)v;
            }
        }
        tf[t] = f;
    }
}

// 8 bf16 of row `row`, zeros outside [0, N); branch-free so a batch of loads can be in flight.
template <int D>
__device__ __forceinline__ u32x4 load_row16_nb(const bf16_t *__restrict__ base, int row, int N, int col) {
    const int rr = min(max(row, 0), N - 1);
    u32x4 v = *reinterpret_cast<const u32x4 *>(base + (size_t)rr * D + col);
    if (rr != row) v = (u32x4){0u, 0u, 0u, 0u};
    return v;
}

// 8 bf16 of the row nearest to `row` inside [0, N): nothing depends on the loaded value, so the
// load stays in flight until its consumer; rows outside the sequence are zeroed by the consumer
// (only tiles at the ends of the sequence have any).
template <int D>
__device__ __forceinline__ u32x4 load_row16_clamped(const bf16_t *__restrict__ base, int row, int N, int col) {
    const int rr = min(max(row, 0), N - 1);
    return *reinterpret_cast<const u32x4 *>(base + (size_t)rr * D + col);
}
__device__ __forceinline__ u32x4 zero_unless(bool keep, u32x4 v) {
    return keep ? v : (u32x4){0u, 0u, 0u, 0u};
}

// LDS transpose read (ds_read_b64_tr_b16): the 16 lanes of a group pass the
// addresses of a 4-row x 16-column block of 16-bit elements (lane p: row p/4,
// columns 4(p%4) .. +3) and lane p gets column p of the 4 rows.  With
// `row0`/`col0` the block origin inside a row-major tile of row stride `stride`
// bytes this yields, for MFMA operands whose k index runs over the tile's rows,
// k = row0 .. row0+3 for column col0 + (lane % 16).
__device__ __forceinline__ bf16x4 lds_read_tr4x16(const unsigned char *tile, int stride, int row0, int col0,
                                                  int n) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const unsigned char *ptr = tile + (row0 + (n >> 2)) * stride + (col0 + 4 * (n & 3)) * 2;
    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(ptr));
    return __builtin_bit_cast(bf16x4, v);
}

// 8 bf16 (16 bytes) of row `row` at element offset `col` of a dense [N][D]
// matrix, zeros when the row is outside [0, N).
template <int D>
__device__ __forceinline__ u32x4 load_row16(const bf16_t *__restrict__ base, int row, int N, int col) {
    u32x4 z = {0u, 0u, 0u, 0u};
    if (row < 0 || row >= N) return z;
    return *reinterpret_cast<const u32x4 *>(base + (size_t)row * D + col);
}

// fp32-arithmetic fallbacks are chosen when this is false.
inline bool mfma_shape_ok(const Problem &p, int in_dt, unsigned flags) {
    return in_dt == CONVATTN_BF16 && !(flags & CONVATTN_FLAG_EXACT) && (p.d == 32 || p.d == 64 || p.d == 128) &&
           p.pk <= kMfmaMaxPk && p.c_q <= 11;
}
// The forward addresses K and V of one (batch, head) through buffer descriptors, which count
// bytes in 32 bits.
// Row / key tiles sit on the z dimension of the grids (at most 65535): the smallest forward tile has
// 88 rows, the backward kernels' tiles 128 rows or keys.
constexpr int kMaxGridZ = 65535;
inline bool mfma_fwd_shape_ok(const Problem &p, int in_dt, unsigned flags) {
    return mfma_shape_ok(p, in_dt, flags) && (size_t)p.Nk * p.d * 2 < (1ull << 31) &&
           ((long long)p.Nq + 87) / 88 <= kMaxGridZ;
}
// The backward kernels put the key taps on one 16-wide MFMA dimension.
inline bool mfma_bwd_shape_ok(const Problem &p, int in_dt, unsigned flags) {
    // (the one-pass kernel addresses Q and dO of one (batch, head) with 32-bit byte offsets)
    // (head dimension 32: the key-stationary kernels only, i.e. not the low-memory dQ pass)
    const bool d32_ok = p.d != 32 || !(flags & CONVATTN_FLAG_LOW_MEMORY);
    return mfma_shape_ok(p, in_dt, flags) && d32_ok && p.c_k <= 15 && (size_t)p.Nq * p.d * 2 < (1ull << 31) &&
           ((long long)p.Nq + 16 + 127) / 128 <= kMaxGridZ && ((long long)p.Nk + 8 + 127) / 128 <= kMaxGridZ;
}

#if defined(__HIPCC__)
// log2 of the dC scale of one (batch, head), taken from D = rowsum(dO o O) of its rows: D is linear
// in dO and of the magnitude of dP, so the power of two s with s |D|max ~ 2^8 keeps the fp16 dC
// tiles (dC = P (dP - D), times s) in fp16's normal range whatever the magnitude of dO is, which
// makes the backward linear in dO.  Every kernel of a backward pass derives the same s from the
// same D.  Called by all `nthreads` threads of a workgroup; `red` is LDS room for one float per
// wave that nothing else uses until the call returns (two barriers inside).
__device__ __forceinline__ float dc_scale_log2_from_d(const float *__restrict__ dl_b, int Nq, int tid, int nthreads,
                                                      float *red) {
    float mx = 0.f;
    for (int i = tid; i < Nq; i += nthreads) mx = fmaxf(mx, fabsf(dl_b[i]));
    mx = wave_max(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = 0.f;
    for (int w2 = 0; w2 < nthreads / 64; ++w2) mx = fmaxf(mx, red[w2]);
    __syncthreads();
    return (mx > 0.f && mx < 3e38f) ? fminf(fmaxf(floorf(8.f - __log2f(mx)), -100.f), 100.f) : 0.f;
}
#endif

#if defined(__HIPCC__)
// {s, log2 s} of a (batch, head) from amax|dO| and amax|V|: s the power of two that brings sqrt(d) amax|dO| amax|V| (a few
// times a typical |dP|) to about 2^12
__device__ __forceinline__ void write_dc_scale(int d, float a, float v, float *out) {
    const float prod = sqrtf((float)d) * a * v;
    float e = 0.f;
    if (prod > 0.f && prod < 3e38f) e = fminf(fmaxf(floorf(12.f - log2f(prod)), -60.f), 60.f);
    out[0] = exp2f(e);
    out[1] = e;
}
#endif

// Raises a kernel's dynamic LDS limit once per device (the attribute is sticky; setting it on every
// launch costs a driver call).  One instance, and one flag word, per kernel instantiation.
template <auto Kern>
inline hipError_t set_max_lds_once(int bytes) {
    static std::atomic<unsigned long long> done{0};   // one bit per device ordinal (mod 64)
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(Kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    return e;
}

// ---- bf16 MFMA kernels ----
hipError_t mfma_fwd(const Problem &p, int out_dt, const void *q, const void *k, const void *v,
                    const float *w, void *o, float *m, float *l, hipStream_t s, float *part = nullptr);
// the same for windows of more than kSparseMaxCk key taps (mfma_fwd calls it)
hipError_t mfma_fwd_wide(const Problem &p, int out_dt, const void *q, const void *k, const void *v,
                         const float *w, void *o, float *m, float *l, hipStream_t s, float *part);
// room for the parts of the query tiles whose keys several workgroups share (`part` above), 0 where none do
size_t mfma_fwd_split_bytes(const Problem &p);

constexpr int kMfmaDqRows = 128;   // query rows per dQ/dW workgroup (= one dW partial)
inline int mfma_dq_tiles(const Problem &p) { return (p.Nq + kMfmaDqRows - 1) / kMfmaDqRows; }
hipError_t mfma_bwd_dq_dw(const Problem &p, int out_dt, const void *q, const void *k, const void *v,
                          const void *d_o, const float *Dl, const float *lse, const float *w, void *dq,
                          float *dw_part, hipStream_t s);

// ---- whole backward with the score chain in registers (bwd_chain3_mfma.hip, bwd_dq_rows.hip) ----
constexpr int kKvKeysPerWg = 128;
inline int mfma_kv_tiles(const Problem &p) { return (p.Nk + 8 + kKvKeysPerWg - 1) / kKvKeysPerWg; }
// The key-stationary kernel's workgroups cover 128 keys each (+ 8:
// the dV ranges start 8 keys early); it leaves one dW partial per workgroup and dS as bf16 blocks
// [key tile of 32][row tile of 32][32 rows][32 keys], which mfma_dq_from_rows multiplies with K.
// dc_scale holds {s, log2 s} per (batch, head): the power of two dC is carried at (mfma_dc_scale).
constexpr int kChainKeys = 32, kChainRows = 32;
// A workgroup walks the row tiles (of 32) that see its keys: under the causal mask those from key block kb's own rows on.
// share > 0: a key block's tiles are cut into parts of at most `share` tiles, one workgroup each (partial dK / dV in
// fp32, added by chain_reduce).  Few (batch, head) pairs or rows leave the launch with less than a round of
// workgroups, as long as its longest one (chain_share has the rule).
struct ChainSpan { int kb, first_rt, len, part, parts; };
__host__ __device__ inline int chain_first_tile(const Problem &p, int kb) {
    return p.causal && kb > 0 ? (kb * kKvKeysPerWg - 8) / kChainRows : 0;
}
__host__ __device__ inline int chain_len(const Problem &p, int kb) { return (p.Nq + kChainRows - 1) / kChainRows - chain_first_tile(p, kb); }
__host__ __device__ inline int chain_parts(const Problem &p, int kb, int share) {
    const int len = chain_len(p, kb);
    return share > 0 && len > share ? (len + share - 1) / share : 1;
}
// workgroup z of a (batch, head)
__host__ __device__ inline ChainSpan chain_span(const Problem &p, int z, int share) {
    ChainSpan s;
    s.kb = z;
    s.part = 0;
    if (share > 0)
        for (s.kb = 0, s.part = z; s.part >= chain_parts(p, s.kb, share); ++s.kb) s.part -= chain_parts(p, s.kb, share);
    s.first_rt = chain_first_tile(p, s.kb);
    s.len = chain_len(p, s.kb);
    s.parts = chain_parts(p, s.kb, share);
    return s;
}
inline int chain_wgs(const Problem &p, int share) {
    int n = 0;
    for (int kb = 0; kb < mfma_kv_tiles(p); ++kb) n += chain_parts(p, kb, share);
    return n;
}
// bytes of the partial dK and dV: [batch, head][workgroup][dK, dV][128 keys][d] fp32
inline size_t chain_part_bytes(const Problem &p, int share) {
    return share > 0 ? (size_t)p.B * p.H * chain_wgs(p, share) * 2 * kKvKeysPerWg * p.d * sizeof(float) : 0;
}
// key blocks with several parts (they are the first ones: the parts do not grow from block to block)
inline int chain_split_blocks(const Problem &p, int share) {
    int n = 0;
    while (n < mfma_kv_tiles(p) && chain_parts(p, n, share) > 1) ++n;
    return n;
}
int chain_share(const Problem &p);
hipError_t chain_reduce(const Problem &p, int out_dt, int share, const float *part, void *dk, void *dv, hipStream_t s);
inline int chain_key_tiles(const Problem &p) { return mfma_kv_tiles(p) * (kKvKeysPerWg / kChainKeys); }
__host__ __device__ inline int chain_row_tiles(const Problem &p) { return (p.Nq + kChainRows - 1) / kChainRows; }
// The dS blocks of one (batch, head) are kept as [key tile][row tile]; under the causal mask key tile kt has
// only the row tiles from kt - 1 on (the rows before them see none of its keys), and only those are kept.
__host__ __device__ inline int chain_ds_first_rt(bool causal, int kt) { return causal && kt > 1 ? kt - 1 : 0; }
// blocks before key tile kt (with kt = the number of key tiles: blocks of a (batch, head))
__host__ __device__ inline long long chain_ds_block_off(bool causal, int n_rt, int kt) {
    if (!causal || kt <= 1) return (long long)kt * n_rt;
    const long long k = kt < n_rt + 1 ? kt : n_rt + 1;   // key tiles from n_rt + 1 on have no blocks
    return k * n_rt - (k - 1) * (k - 2) / 2;
}
inline size_t chain_ds_bytes(const Problem &p) {
    return (size_t)p.B * p.H * (size_t)chain_ds_block_off(p.causal != 0, chain_row_tiles(p), chain_key_tiles(p)) *
           kChainKeys * kChainRows * 2;
}
// {s, log2 s} per (batch, head) followed by 32 x 2 partial maxima per (batch, head)
inline size_t chain_scale_bytes(const Problem &p) { return (size_t)p.B * p.H * (2 + 64) * sizeof(float); }
hipError_t mfma_dc_scale(const Problem &p, const void *d_o, const void *v, float *dc_scale, hipStream_t s);
// its second step alone; D, LSE and the dC scale together (reduce_kernels.hip)
constexpr int kScaleChunks = 32;
hipError_t dc_scale_finish(const Problem &p, float *dc_scale, hipStream_t s);
hipError_t bwd_prepare(const Problem &p, int out_dt, const void *o, const void *d_o, const void *v, const float *m, const float *l,
                       float *D, float *lse, float *dc_scale, hipStream_t s);
// want: bit 0 = dK and dV, bit 1 = dS blocks (for dQ) and the dW partial; dc_scale may be null when
// bit 1 is clear (the kernel then takes the scale from D).
#define CHAIN_DECL(name)                                                                                   \
    hipError_t name(const Problem &p, int out_dt, const void *q, const void *k, const void *v, const void *d_o, \
                    const float *Dl, const float *lse, const float *w, const float *dc_scale, void *dk, void *dv, \
                    void *ds_ws, float *dw_part, int share, float *kv_part, hipStream_t s)
CHAIN_DECL(mfma_bwd_chain3_kv);
CHAIN_DECL(mfma_bwd_chain3_qw);
CHAIN_DECL(mfma_bwd_chain3_all);
CHAIN_DECL(mfma_bwd_chain3_split);   // everything, with share > 0
#undef CHAIN_DECL
inline hipError_t mfma_bwd_chain(const Problem &p, int out_dt, int want, const void *q, const void *k, const void *v,
                                 const void *d_o, const float *Dl, const float *lse, const float *w,
                                 const float *dc_scale, void *dk, void *dv, void *ds_ws, float *dw_part,
                                 hipStream_t s, int share = 0, float *kv_part = nullptr) {
    if (want == 1) return mfma_bwd_chain3_kv(p, out_dt, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s);
    if (want == 2) return mfma_bwd_chain3_qw(p, out_dt, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s);
    if (share) return mfma_bwd_chain3_split(p, out_dt, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s);
    return mfma_bwd_chain3_all(p, out_dt, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s);
}
// What follows the key-stationary kernel: dQ, the sum of the n_wg dW partials per (batch, head) and, with share > 0, dK and dV from
// their parts.  One launch where dQ's waves share keys (small problems), else one each.
hipError_t mfma_bwd_products(const Problem &p, int out_dt, const void *k, const void *ds_ws, const float *dc_scale, int n_wg,
                             const float *dw_part, int share, const float *kv_part, void *dq, void *dk, void *dv, float *dw,
                             hipStream_t s);
// heads_inner: the blocks lie [batch][block][head] (all heads of a block side by side) instead of [batch, head][block]
hipError_t mfma_dq_from_rows(const Problem &p, int out_dt, const void *k, const void *ds_ws,
                             const float *dc_scale, void *dq, hipStream_t s, bool heads_inner = false);

// ---- decode as an HBM stream (decode_stream.hip) ----
bool decode_stream_ok(const Problem &p, int in_dt, unsigned flags);
// Where the decode kernel finds K and V rows beyond Problem's batch / head strides.
struct KvArgs {
    const int *table;       // block table [B][table_stride] of page numbers, or null: contiguous rows
    const int *seq_lens;    // keys per batch entry [B] (clamped to Problem::Nk), or null: Nk for all
    long long page_stride;  // elements between pages of the pool
    int table_stride;
    int page_shift;         // log2 of the keys per page
    int group;              // query heads per KV head (>= 1)
};
// query heads that share KV heads in pairs or fours, d = 64 or 128 (decode_shared.hip)
hipError_t decode_shared(const Problem &p, const KvArgs &kv, const void *q, const void *k, const void *v, const float *w,
                         float *o_part, float *m_part, float *l_part, hipStream_t s);
hipError_t decode_stream_kv(const Problem &p, const KvArgs &kv, const void *q, const void *k, const void *v,
                            const float *w, float *o_part, float *m_part, float *l_part, hipStream_t s);
hipError_t decode_stream(const Problem &p, const void *q, const void *k, const void *v, const float *w,
                         float *o_part, float *m_part, float *l_part, hipStream_t s);
// a step's split count (ragged: the entries of the batch have lengths of their own)
int decode_splits(long long heads, int Nk, bool ragged, int d);
int decode_step_splits(long long heads, int Nk, int d, int asked);
// The whole step in one launch, where decode_whole_waves is not 0
int decode_whole_waves(const Problem &p);
hipError_t decode_whole(Problem p, int out_dt, const void *q, const void *k, const void *v, const float *w, void *o, float *m, float *l,
                        hipStream_t s);

}  // namespace convattn
