// Pieces of the key-stationary backward kernel (bwd_chain3_mfma.hip): LDS layout,
// fragment addressing, DPP row windows, Toeplitz bands for the packed operand order, the argument block.
#pragma once
#include <type_traits>

#include "mfma_common.hpp"

namespace convattn {
namespace chain {

constexpr int NP = 4;            // wave triples = 32-key ranges per workgroup
constexpr int WK = 32;           // own keys per triple
constexpr int BKW = NP * WK;     // 128 keys per workgroup
constexpr int BR = 32;           // query rows per tile
constexpr int NCB = 3;           // C / dP / dC blocks: keys c0-8+16cb
constexpr int NDB = 2;           // dS blocks: keys c0+16sb
constexpr int SST = 104;         // bytes per row of the S tile in LDS (48 keys fp16 + 8)
constexpr int S_RING = 72;       // rows of the S ring: a tile being written, the tile before it and 8 rows more (>= c_q - 1)
constexpr int CST = 104;         // bytes per row of the dC tile (48 keys fp16 + 8)
constexpr int PST = 72;          // bytes per row of the P and dS tiles (32 keys bf16 + 8)
static_assert(BKW == kKvKeysPerWg && WK == kChainKeys && BR == kChainRows, "dS workspace layout");

// The bands of the sparse products (two tap slots each, see SparseTaps).  The half of a fragment that belongs to one slot is the same
// wherever that slot stands: a row of 32 lanes x 16 bytes, and a product whose two slots have neighbouring rows reads its
// fragment as 1 KB from the first one's row on.  Even CQT: two more rows for the product of slots 0 and CQT - 1.  Odd: two more for each
// parity's single slot, the operand of a dense product (64 lanes x 16 bytes, the window's first block in the even dwords).  `flip`: the
// transposed convolution, whose rows are counted downwards (row offset e = delta + CQT - 1, tap slot CQT - 1 - slot).
template <int CQT> using ChainTaps = SparseTaps<CQT>;
template <int CQT> struct ChainBands {
    using T = ChainTaps<CQT>;
    static constexpr int rows = CQT + (T::odd ? 4 : 2), row_bytes = 512;
    static constexpr int slot(int row) {
        return row < CQT ? row : T::odd ? T::single_slot(row >= CQT + 2) : row == CQT ? 0 : CQT - 1;
    }
    // first row of product i of output parity ob, and of its single slot
    static constexpr int row(int i, int ob) { return T::odd ? 2 * i + ob : !ob && i == T::products - 1 ? CQT : 2 * i + 1 - ob; }
    static constexpr int single_row(int ob) { return CQT + 2 * ob; }
    static constexpr bool rows_right() {
        for (int ob = 0; ob < 2; ++ob)
            for (int i = 0; i < T::products; ++i)
                for (int half = 0; half < 2; ++half)
                    if (T::slot(T::tuple(i, ob), half, ob) != slot(row(i, ob) + half)) return false;
        return true;
    }
    static_assert(T::every_slot_once() && rows_right(), "rows of the products");
    // this lane's 16 bytes of a row
    static __device__ __forceinline__ f16x8 frag(int row, const float *__restrict__ w_head, int c_q, int c_k, int pk, int g, int n,
                                                 bool flip, float mul) {
        const int t = flip ? CQT - 1 - slot(row) : slot(row), a = t - (CQT - c_q);
        const bool single = T::odd && row >= CQT;
        // (unconditional loads from clamped indices: the eight of a fragment are in flight together)
        const float *w = w_head + min(max(a, 0), c_q - 1) * c_k;
        float v[8];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int kappa = single ? 8 * ((row - CQT) & 1) + 4 * (g & 1) + 2 * (q >> 1) : sparse_key(g, q);
                const int off = kappa + e + ((single ? (q & 1) == 0 : kappa + 1 > n) ? 0 : 16) - kKeyHalo - n;
                const int bb = flip ? pk - off : pk + off;
                v[2 * q + e] = w[min(max(bb, 0), c_k - 1)];
                if (a < 0 || bb < 0 || bb >= c_k) v[2 * q + e] = 0.f;
            }
        f16x8 f;
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (_Float16)(v[e] * mul);
        return f;
    }
    // c + the single slot of parity ob, from the tuple it is in (`swapped`: the window's first block in the odd dwords)
    static __device__ __forceinline__ f32x4 single(f16x8 band, int ob, bool swapped, u32x8 rows, f32x4 c) {
        const u32x4 v = ob ? (u32x4){rows[4], rows[5], rows[6], rows[7]} : (u32x4){rows[0], rows[1], rows[2], rows[3]};
        return mfma_f16(band, __builtin_bit_cast(f16x8, swapped ? (u32x4){v[1], v[0], v[3], v[2]} : v), c);
    }
    // the rows from `first` on to LDS, dealt out in pairs to `n_waves` waves
    static __device__ __forceinline__ void build(unsigned char *tab, int first, const float *__restrict__ w_head, int c_q, int c_k, int pk,
                                                 bool flip, float mul, int wave, int n_waves, int g, int n) {
        for (int r0 = first + 2 * wave; r0 < rows; r0 += 2 * n_waves) {
            const int r = r0 + (g >> 1);
            const f16x8 f = frag(r, w_head, c_q, c_k, pk, g, n, flip, mul);
            if (r < rows) *reinterpret_cast<f16x8 *>(tab + (r - first) * row_bytes + ((g & 1) * 16 + n) * 16) = f;
        }
    }
};

template <int D, int CQT> struct ChainLds {
    // Q / dO tiles are filled by buffer loads with the LDS modifier (64 lanes = 1 KB of consecutive
    // LDS), which rules out padded rows.  A tile of 32 rows is kept as [k-step ks][row parity f]
    // [row pair n][64 bytes]: the 4 chunks of 16 bytes that row 2n + f holds of head-dim columns
    // 32 ks .. 32 ks + 31, chunk c at position c ^ (n / 4 mod 4).  Row fragments (lane n reads row
    // 2n + f) and transposed fragments then touch every bank equally often, and k-step, parity and
    // head-dim block are constant offsets from one lane address.
    static constexpr int RST = D * 2;                               // bytes per Q / dO row
    // (a plane of one parity is 32 bytes longer than its rows: the transpose reads take two rows of either parity at a time)
    static constexpr int plane = 1024 + 32, tile_bytes = RST / 32 * plane;
    static constexpr int q_off = 0, q_slots = 4;                    // tiles it-2 .. it+1
    static constexpr int g_off = q_off + q_slots * tile_bytes, g_slots = 3;  // tiles it-1 .. it+1
    static constexpr int stat_off = g_off + g_slots * tile_bytes;   // LSE and D of a tile: two slots
    static constexpr int stat_bytes = 2 * (2 * BR * 4);
    // the bands of the convolution, then those of the transposed one that the key waves do not keep in registers: those
    // from product key_regs on (up to d = 64 and up to 6 slots none; 8 slots at d = 128 all, 11 what leaves room for the S ring)
    using Bands = ChainBands<CQT>;
    static constexpr int key_regs = D <= 64 || CQT <= 6 ? Bands::T::products : CQT <= 8 ? 0 : 2;
    static constexpr int key_row = 2 * key_regs;   // first row of the transposed bands in LDS
    static constexpr int key_rows = key_regs < Bands::T::products ? Bands::rows - key_row : 0;
    static constexpr int band_off = stat_off + stat_bytes;
    static constexpr int key_band_off = band_off + Bands::rows * Bands::row_bytes;
    static constexpr int band_bytes = (Bands::rows + key_rows) * Bands::row_bytes;
    static_assert(key_regs == 0 || key_regs == Bands::T::products || Bands::T::odd, "rows of product i from 2 i on");
    static constexpr int pair_off = band_off + band_bytes;
    static constexpr int ring_rows = CQT > 9 ? S_RING + 2 : S_RING;   // >= 64 + CQT - 1
    static constexpr int s_bytes = ring_rows * SST;
    static constexpr int c_bytes = 2 * BR * CST;
    static constexpr int p_bytes = 2 * BR * PST;
    static constexpr int ds_bytes = BR * PST;
    static constexpr int pair_bytes = s_bytes + c_bytes + p_bytes + ds_bytes;
    // V and, where there is room, K fragments of the block after the workgroup's keys (16 rows each): the wave that computes it has no
    // registers to keep them in (with K in registers 12 and 24 spilled at d = 128, 6 and 8 slots, now 0 and 2, in parts 0 and 16; kernel of B4 H16 N4096 1254 ->
    // 1253 and 1384 -> 1352 us, of B1 H32 N16384 6x11 9075 -> 9009)
    static constexpr int e_off = pair_off + NP * pair_bytes;
    static constexpr bool k_park = D == 128 && CQT <= 8;   // (11 slots: no room)
    static constexpr int total = e_off + 16 * D * 2 * (k_park ? 2 : 1);
    static_assert(CQT * 2 * 1024 <= NP * pair_bytes, "room for the dW accumulators (they take the place of the pairs' tiles)");
};

// A lane-dependent LDS offset the compiler may not fold or hoist: what is added to it afterwards
// stays a constant and ends up in the instructions' offset fields instead of one address register
// per fragment.
__device__ __forceinline__ unsigned int opaque(unsigned int x) {
    asm volatile("" : "+v"(x));
    return x;
}

__device__ __forceinline__ bf16x4 lds_tr64(const unsigned char *ptr) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(ptr));
    return __builtin_bit_cast(bf16x4, v);
}
// Transposed fragment of a row-major tile of 16-bit elements with `stride` bytes per row:
// k = rows 4g .. 4g+3 then 16+4g .. 16+4g+3, column col0 + n.  `lane_ptr` is the tile's address plus
// tr_lane_off(stride, g, n).
__device__ __forceinline__ unsigned int tr_lane_off(int stride, int g, int n) {
    return (4 * g + (n >> 2)) * stride + 4 * (n & 3) * 2;
}
__device__ __forceinline__ bf16x8 read_tr(const unsigned char *lane_ptr, int stride, int col0) {
    bf16x4 lo = lds_tr64(lane_ptr + col0 * 2);
    bf16x4 hi = lds_tr64(lane_ptr + 16 * stride + col0 * 2);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int CTRL>
__device__ __forceinline__ unsigned int dpp_keep(unsigned int old, unsigned int src) {
    return (unsigned int)__builtin_amdgcn_update_dpp((int)old, (int)src, CTRL, 0xf, 0xf, false);
}
// A DPP move that writes every lane (rotations): no previous value to keep.
template <int CTRL>
__device__ __forceinline__ unsigned int dpp_mov(unsigned int src) {
    return (unsigned int)__builtin_amdgcn_mov_dpp((int)src, CTRL, 0xf, 0xf, true);
}
// Lane n of a row of 16 gets cur[n - S] for n >= S and prev[16 + n - S] below: a window that
// starts S lanes before `cur` in the sequence prev | cur.
template <int S>
__device__ __forceinline__ unsigned int win_up(unsigned int prev, unsigned int cur) {
    if constexpr (S == 0) {
        return cur;
    } else {
        const unsigned int x = dpp_mov<0x120 + S>(prev);  // row_ror:S
        return dpp_keep<0x110 + S>(x, cur);               // row_shr:S, lanes below S keep x
    }
}
// Lane n gets a[n + S] for n + S < 16 and b[n + S - 16] above: a window that starts S lanes into
// `a` in the sequence a | b.
template <int S>
__device__ __forceinline__ unsigned int win_down(unsigned int a, unsigned int b) {
    if constexpr (S == 0) {
        return a;
    } else {
        const unsigned int x = dpp_mov<0x120 + 16 - S>(b);  // row_ror:(16-S)
        return dpp_keep<0x100 + S>(x, a);                   // row_shl:S, the last S lanes keep x
    }
}

__device__ __forceinline__ unsigned int pack_f16_rtz(float a, float b) {
    return __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(a, b));
}

// Kernel arguments as one block: each role reads them from the kernel argument segment with
// scalar loads (arguments of a device function would arrive in vector registers).
struct ChainArgs {
    Problem p;
    const bf16_t *Q, *K, *V, *dO;
    const float *Dl, *LSE, *W, *dc_scale;
    void *dK, *dV;
    bf16_t *dS_ws;
    float *dW_part;
    int n_rt, share;    // share, kv_part: see ChainSpan
    float *kv_part;
};

// The kernel argument segment lives in the constant address space; host passes of the compiler
// do not know that attribute.
#if defined(__HIP_DEVICE_COMPILE__)
#define CHAIN_CONST_AS __attribute__((address_space(4)))
#else
#define CHAIN_CONST_AS
#endif

}  // namespace chain
}  // namespace convattn
