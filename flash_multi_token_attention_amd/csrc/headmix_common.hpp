// Pieces shared by the head-mixing kernels that work on tiles of (row, key) pairs of all heads
// (headmix_probs.hip: forward, headmix_scores.hip: backward).
//
// A workgroup owns R query rows of all heads of a batch entry and walks KT keys per step, alternating between
// "a wave takes heads" (products of rows, bf16 MFMA) and "a wave takes rows" (the head mix as a product over the head
// index on the fp32 MFMA); the two meet in LDS arrays [head][tile row][key].  What the tiles leave
// (probabilities, dS) goes to global memory as bf16 blocks of 32 rows x 32 keys in the layout of the
// product kernels, [row parity][key half][row pair][16 keys], the blocks of all heads side by side:
// [batch][block][head].
#pragma once
#include "mfma_common.hpp"

namespace convattn {
namespace headmix {

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// Workgroup barrier for data that is exchanged through LDS: waits for this wave's LDS operations, not for the
// global loads it has issued ahead.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// the value of the lane ROR places on in the row of 16
template <int ROR> __device__ __forceinline__ float row16_rot(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + ROR, 0xf, 0xf, true));
}

// base (the same in all lanes) + a lane's byte offset: the form the loads and stores take with the base in scalar registers
template <typename V> __device__ __forceinline__ const V *at(const bf16_t *base, unsigned off) {
    return reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + off);
}
template <typename V> __device__ __forceinline__ V *at(bf16_t *base, unsigned off) {
    return reinterpret_cast<V *>(reinterpret_cast<char *>(base) + off);
}

constexpr int kBlock = kChainRows * kChainKeys;   // elements of a block

// H heads, WAVES waves, R rows; 64 pairs per wave in the mixing phase: lane n = RW rows x NQ quads of keys.
template <int H_, int WAVES_, int R_> struct Tile {
    static constexpr int H = H_, WAVES = WAVES_, R = R_, RB = R / 16, KT = WAVES * 64 / R, KB = KT / 16, NQ = KT / 4;
    static constexpr int RW = R / WAVES, HPW = H / WAVES, HB = H / 16;
    static_assert(RW * NQ == 16 && HPW >= 1 && (NQ == 4 || NQ == 8), "64 pairs per wave");
    static constexpr int HS = R * KT + 4;                   // floats per head (+4: 16 heads on 16 bank quads)
    static constexpr int arr = H * HS;                      // floats of one array
    static constexpr int WST = H + 4;                       // floats per row of w in LDS
    // Four keys 4q .. 4q+3 of tile row `lr` sit at float lr * KT + 4 * slot: the XOR spreads both the score
    // phase's writes (16 rows, one quad) and the mixing phase's reads (RW rows, all quads) over all banks.
    __device__ static __forceinline__ int slot(int lr, int q) { return q ^ ((lr >> (NQ == 4 ? 2 : 1)) & (NQ - 1)); }
    // Query row of tile row lr: even rows of the 32-row block first, as the blocks are laid out
    __device__ static __forceinline__ int row(int i0, int lr) {
        return RB == 2 ? i0 + 2 * (lr & 15) + (lr >> 4) : i0 + 2 * (lr & 7) + (lr >> 3);
    }
};

// The work of a launch: the key steps of all row tiles of all batch entries laid end to end, cut into even shares, one
// per workgroup; a share's part of a row tile is a segment.  One round of workgroups, all done at the same time:
// chunks of keys per row tile left the CUs with up to 335 of 258 steps at B4 H16 N4096 (55 of 33 at B2 H32 N2048), the
// causal tiles being of all lengths and a launch five rounds.  Row tiles lie in pairs last, first, last but
// one, second, ..: the pairs are equally long under the causal mask, so that where a share is about a pair (or a
// simple fraction of one) neighbours walk the same keys at the same time.
struct Plan {
    int n_tiles, unit, split_shift;   // row tiles of a batch entry; key steps per 32 keys; log2 of the row tiles per 32 rows
    int pair_len, entry_len;          // steps of a pair of row tiles, of a batch entry
    int share, n_wg, max_segments;    // steps per workgroup, workgroups, segments of a row tile at most
    int causal, n_rt32, B;

    __host__ __device__ int len(int rt) const { return (causal ? (rt >> split_shift) + 1 : n_rt32) * unit; }
    // position of row tile rt of batch entry b
    __host__ __device__ int start(int b, int rt) const {
        const int p = n_tiles - 1 - rt, first = p <= rt ? p * pair_len : rt * pair_len + len(p);
        return b * entry_len + first;
    }
};
template <typename T> Plan make_plan(int B, int N, int causal) {
    Plan p;
    p.n_rt32 = (N + 31) / 32;
    p.causal = causal;
    p.B = B;
    p.unit = 32 / T::KT;
    p.split_shift = T::R == 16;
    p.n_tiles = p.n_rt32 << p.split_shift;
    p.pair_len = p.len(0) + p.len(p.n_tiles - 1);
    p.entry_len = p.n_tiles / 2 * p.pair_len + (p.n_tiles & 1 ? p.len(p.n_tiles / 2) : 0);
    const long long total = (long long)B * p.entry_len;
    p.share = (int)((total + 255) / 256);
    p.n_wg = (int)((total + p.share - 1) / p.share);
    p.max_segments = (p.len(p.n_tiles - 1) + p.share - 1) / p.share + 1;
    return p;
}
// Neighbouring shares run on the same XCD (workgroup ids go round robin over the eight): the rows of K and V that
// they walk come from one L2.
__device__ __forceinline__ int share_of_workgroup(const Plan &pl) {
    const int per = (pl.n_wg + 7) / 8, w = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    return (int)(blockIdx.x >> 3) < per && w < pl.n_wg ? w : -1;
}
inline int plan_grid(const Plan &pl) { return (pl.n_wg + 7) / 8 * 8; }
// A segment: steps s0 .. s_end-1 of row tile rt of batch entry b.  A workgroup takes them in the order step(0),
// step(1), ..: rotated, so that at a time t all workgroups are at key steps of the residue t modulo the share, i.e. at few
// different keys (from s0 on, segments beginning anywhere, the workgroups of an XCD found 10 % of the rows of K
// and V in its L2; rotated, 78 and 66 % of all accesses of the forward and the backward hit, B4 H16 N4096 d128).
// `down` (long shares of the backward, score_plan): a segment that ends with its share, and does not begin with it, is
// walked from its last step down.  The shares end at the same time, so at a time t those on the short tiles of an entry
// are all at the step that many from the start, whatever their lengths; rotated, neighbours are two steps apart, and the
// blocks that are written meanwhile (1 MB per step on an XCD) push the rows out of the L2.
struct Segment {
    int b, rt, s0, s_end, rot;
    bool down;
    __device__ __forceinline__ int len() const { return s_end - s0; }
    __device__ __forceinline__ int step(int i) const {
        if (down) return s_end - 1 - i;
        const int s = s0 + rot + i;
        return s >= s_end ? s - (s_end - s0) : s;
    }
};
// the one at position x of share `id`
__device__ __forceinline__ Segment find_segment(const Plan &pl, int id, int x, bool down) {
    const int begin = id * pl.share;
    const int end = (int)min((long long)begin + pl.share, (long long)pl.entry_len * pl.B);
    Segment sg;
    sg.b = __builtin_amdgcn_readfirstlane(x / pl.entry_len);
    const int r = x - sg.b * pl.entry_len, p = __builtin_amdgcn_readfirstlane(r / pl.pair_len);
    sg.s0 = r - p * pl.pair_len;
    sg.rt = pl.n_tiles - 1 - p;
    const int first = pl.len(sg.rt);
    if (sg.s0 >= first) { sg.s0 -= first; sg.rt = p; }
    sg.s_end = min(pl.len(sg.rt), sg.s0 + end - x);
    int rot = (x - begin - sg.s0) % pl.share;
    rot = __builtin_amdgcn_readfirstlane(rot < 0 ? rot + pl.share : rot);
    sg.rot = rot < sg.len() ? rot : 0;
    sg.down = down && __builtin_amdgcn_readfirstlane(x > begin && x + sg.len() == begin + pl.share) != 0;
    return sg;
}

// Row fragments (lane 16g + n: tile row 16 rb + n, columns 32 ks + 8g ..) of rows i0 .. i0+R-1 of a head: whole rows
// loaded, turned in `st`, this wave's room of R * (2 D + 16) bytes in LDS.  Rows past the last: copies of it.
template <typename T, int D>
__device__ __forceinline__ void turn_rows(bf16x8 (&f)[T::RB][D / 32], const bf16_t *__restrict__ src, int i0, int N, unsigned char *st) {
    constexpr int CPR = D / 8, RST = D * 2 + 16, LD = T::R * CPR / 64;
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    u32x4 raw[LD];
#pragma unroll
    for (int i = 0; i < LD; ++i) {
        const int c = lane + i * 64;
        raw[i] = *reinterpret_cast<const u32x4 *>(src + (size_t)min(i0 + c / CPR, N - 1) * D + (c % CPR) * 8);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < LD; ++i) {
        const int c = lane + i * 64;
        *reinterpret_cast<u32x4 *>(st + (c / CPR) * RST + (c % CPR) * 16) = raw[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int rb = 0; rb < T::RB; ++rb)
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks)
            f[rb][ks] = *reinterpret_cast<const bf16x8 *>(st + T::row(0, rb * 16 + n) * RST + ks * 64 + g * 16);
}

// Rows of a tensor in the order in which the score phases' lanes read them: [batch, head][16 rows][k step][lane][8]
// (lane 16g + n: row n, columns 32 ks + 8g ..), zeros past the last row.  Read straight from the rows, a fragment
// load has neighbouring lanes in different rows: 64 cache accesses instead of 16, and the backward's score kernel was
// bound by them (3.3 M of its 4.1 M clocks per CU at B4 H16 N4096 d128).  One copy of K and V (0.04 ms there) is read
// N / 32 times.  V may be null.
template <int D>
__device__ __forceinline__ void frag_order(size_t f, int N, int n_t16, const bf16_t *__restrict__ K, const bf16_t *__restrict__ V,
                                           bf16_t *__restrict__ KF, bf16_t *__restrict__ VF, size_t n_frag) {
    if (f >= n_frag) return;   // (one 1 KB fragment per wave)
    constexpr int KS = D / 32;
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const size_t bh = f / ((size_t)n_t16 * KS);
    const int r = (int)(f - bh * n_t16 * KS), row = (r / KS) * 16 + n, col = (r % KS) * 32 + 8 * g;
    *reinterpret_cast<u32x4 *>(KF + f * 512 + lane * 8) = load_row16<D>(K + bh * N * D, row, N, col);
    if (V) *reinterpret_cast<u32x4 *>(VF + f * 512 + lane * 8) = load_row16<D>(V + bh * N * D, row, N, col);
}
inline size_t frag_count(int BH, int N, int d) { return (size_t)BH * ((N + 31) / 32 * 2) * (d / 32); }

}  // namespace headmix
}  // namespace convattn
