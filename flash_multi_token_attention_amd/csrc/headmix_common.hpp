// Pieces shared by the head-mixing kernels that work on tiles of (row, key) pairs of all heads
// (headmix_probs.hip: forward, headmix_scores.hip: backward).
//
// A workgroup owns R query rows of all heads of a batch entry and walks KT keys per step, alternating between
// "a wave takes heads" (products of rows, bf16 MFMA) and "a wave takes rows" (the head mix as a product over the head
// index with fp32's precision); the two meet in LDS arrays [head][tile row][key].  What the tiles leave
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

// The mix of 32 heads on the bf16 MFMA: every operand is the sum of three bf16 numbers, x = hi + mid + lo exactly (8 significant
// bits each, rounded to nearest), and six of the nine products are taken; each of the others is below 2^-26 |a b|.  96 clocks for a
// contraction over 32 heads where the fp32 MFMA takes 256; that was 60 % of the time of headmix_scores_kernel<32, 64>, whose vector ALUs
// were 7 % busy.  B2 H32 N2048 d64, us: scores 346 -> 305, probabilities 170 -> 152; B2 H32 N1500 d32 182 -> 157 and 89 -> 82; d128 252 -> 248
// and 119 -> 110.  log L of the forward against 64 bits, means of 12 seeds: 1.616e-8 -> 1.580e-8 of its norm (N500 d64), 1.520 -> 1.480e-8 (N330 d128), its
// gradients as before.  With 16 heads three of five clocks stay and the matrix pipe does not bind.  dw (a sum over pairs, whose operands
// would both have to be split) stays on the fp32 MFMA: 305 us, on this one 311.
// Infinities and NaN leave a NaN in a rest, so in every head's sum: such a step is repeated on the fp32 MFMA (has_nan).
struct Split { bf16x8 hi, mid, lo; };
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(unsigned, (bf16x2){(__bf16)a, (__bf16)b});
}
__device__ __forceinline__ Split split8(const float (&v)[8]) {
#pragma clang fp contract(off)   // (a product whose rest is taken would be computed again, its factors kept)
    u32x4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = v[2 * i], b = v[2 * i + 1];
        h[i] = bf16_pair(a, b);
        a -= __uint_as_float(h[i] << 16);
        b -= __uint_as_float(h[i] & 0xffff0000u);
        m[i] = bf16_pair(a, b);
        a -= __uint_as_float(m[i] << 16);
        b -= __uint_as_float(m[i] & 0xffff0000u);
        l[i] = bf16_pair(a, b);
    }
    return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}
// The split of a 32 x 32 matrix in LDS as A operands [hi, mid, lo][16 rows][lane][8]: lane (g, n) row n, k slot 4y + s of its eight = column
// 16y + 4g + s, the heads of the fp32 path's accumulators
constexpr int kSplitBytes = 3 * 2 * 64 * 16;
__device__ __forceinline__ void put_split(void *dst, int row, int col, float v) {
    unsigned short *p = static_cast<unsigned short *>(dst) + ((row >> 4) * 64 + ((col >> 2) & 3) * 16 + (row & 15)) * 8 + (col >> 4) * 4 + (col & 3);
#pragma unroll
    for (int part = 0; part < 3; ++part) {
        const unsigned u = bf16_pair(v, 0.f) & 0xffffu;
        p[part * 1024] = (unsigned short)u;
        v -= __uint_as_float(u << 16);
    }
}
template <int HB> __device__ __forceinline__ bool has_nan(const f32x4 (&z)[HB][4]) {
    bool nan = false;
#pragma unroll
    for (int x = 0; x < HB; ++x)
#pragma unroll
        for (int t = 0; t < 4; ++t) nan |= __builtin_isunordered(z[x][t][0], z[x][t][1]) | __builtin_isunordered(z[x][t][2], z[x][t][3]);
    return __any(nan);
}
// c[x][u] += A_x B_u for both 16 rows x of the matrix at `a`, the small products first.  (A part of the matrix is read when its
// products are due: registers are short.)
template <int U>
__device__ __forceinline__ void mfma_split(f32x4 *const (&c)[2], const void *a, int lane, const Split (&b)[U]) {
    const bf16x8 *p = static_cast<const bf16x8 *>(a) + lane;
#pragma unroll
    for (int part = 2; part >= 0; --part) {
        asm volatile("" ::: "memory");
        const bf16x8 w[2] = {p[part * 128], p[part * 128 + 64]};
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (part == 0) c[x][u] = mfma_bf16(w[x], b[u].lo, c[x][u]);
                if (part <= 1) c[x][u] = mfma_bf16(w[x], b[u].mid, c[x][u]);
                c[x][u] = mfma_bf16(w[x], b[u].hi, c[x][u]);
            }
    }
}

// z[x][t] += (the 32 x 32 matrix in `w`) S for the keys t of the lane's tile row, the heads in the order of put_split
template <typename T>
__device__ __forceinline__ void mix_split(f32x4 (&z)[T::HB][4], const float *S, int pos, int g, const void *w, int lane) {
#pragma unroll
    for (int t = 0; t < 4; t += 2) {   // (two keys at a time; four: 314 us where this is 305, one: 319, the matrix is read more often)
        float2 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const float2 *>(S + (16 * (i >> 2) + 4 * g + (i & 3)) * T::HS + pos + t);
        const Split sp[2] = {split8({v[0].x, v[1].x, v[2].x, v[3].x, v[4].x, v[5].x, v[6].x, v[7].x}),
                             split8({v[0].y, v[1].y, v[2].y, v[3].y, v[4].y, v[5].y, v[6].y, v[7].y})};
        mfma_split<2>({&z[0][t], &z[T::HB - 1][t]}, w, lane, sp);
    }
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
