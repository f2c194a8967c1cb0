// Training forward of conv-attention on bf16 MFMA (gfx950): the scores never leave the registers.
//
// Workgroup = 4 waves of one (batch, head); a wave computes scores for 32 consecutive query rows
// (the first CQT-1 of them only as the window's halo above its 33-CQT output rows) and keeps
// O^T, the row sums and the softmax bases of its rows in registers for the whole key loop.
// Lane n of score fragment f holds row base + 2n + f.  Per 32-key step:
//   1. all waves issue the loads of the next step's K / V rows, which go from global memory
//      straight into the LDS buffer the step before this one has just left (buffer loads with the
//      LDS modifier: no staging registers, no LDS writes by the waves; a tile is kept as
//      [k-step][row][64 bytes] with the four 16-byte chunks XOR-swizzled with the row index, so that
//      one lane address per matrix serves every fragment; one barrier per step);
//   2. S^T = K Q^T for two 16-key blocks; the accumulator layout (lane = query row, 4 keys per
//      lane group) is, packed to fp16 after the causal pre-mask, already the B operand layout of
//      the convolution MFMA: a window of 32 input keys is two packed blocks side by side in a lane
//      and the output block sits 8 keys into it.  The last block of a step stays for the next
//      step; no score is computed twice along the keys;
//   3. convolution: C^T += T_a^T S^T(rows shifted by the tap), two taps per sparse product (SparseTaps).
//      A shift by an even number of rows is a DPP row shift of the packed registers, by an odd number
//      the other fragment shifted; rows shifted in from above the wave's first row are zeros and only
//      reach halo rows.  A block's shifted rows are made once and kept for both windows it is in.
//      What bounds the kernel is the issue of vector instructions (63 % of the cycles at B4 H16 N4096 d64 6x11)
//      beside the matrix pipe (52 %), at a clock of 1.8 GHz.  Dense products of one tap each, whose windows were
//      shifted anew and whose bands every lane gathered from memory, against these, us: B4 H16 N4096 6x11 d128
//      440 -> 392, N2048 d64 88 -> 75, B1 H32 N5399 d64 11x11 452 -> 360, B4 H16 N4096 d64 7x7 357 -> 299, B1 H32 N4096 d64
//      3x3 119 -> 110, B2 H8 N526 d32 6x11 14.5 -> 11.9;
//   4. post-mask (-inf) and softmax numerators against a per-row base that is only raised (with
//      a rescale of O and the row sums) when a score exceeds it by more than 2^6: no cross-lane
//      traffic otherwise.  The true row maximum is kept per lane, relative to the base, for the M output;
//   5. O^T += V^T P^T: V^T fragments through the LDS transpose read, P^T straight from the
//      softmax registers.
#include "mfma_common.hpp"

namespace convattn {
namespace {


// DPP move (CTRL 0x110+s: row_shr:s, lane n of a row of 16 gets lane n-s); lanes without a
// source lane get 0.
template <int CTRL>
__device__ __forceinline__ unsigned int dpp_zero(unsigned int src) {
    return (unsigned int)__builtin_amdgcn_update_dpp(0, (int)src, CTRL, 0xf, 0xf, true);
}

__device__ __forceinline__ unsigned int opaque_u32(unsigned int x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ bf16x4 lds_tr64(__attribute__((address_space(3))) const unsigned char *ptr) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(ptr));
    return __builtin_bit_cast(bf16x4, v);
}

constexpr int NW = 4;             // waves per workgroup
constexpr int BK = 32;            // keys per step
constexpr float kMaxSlack = 6.f;  // log2 units a score may exceed its row's exponent base by
// A wave computes scores for 32 consecutive rows; the first CQT-1 of them are only the
// window's halo, the other 33-CQT are its output rows.
constexpr int wave_rows(int cqt) { return 33 - cqt; }

constexpr int kFwdPfv = 2;    // V^T fragments read ahead of their MFMAs in the P V phase
template <int D> struct FwdLds {
    // K / V rows go from global memory straight into LDS (buffer loads with the LDS modifier: the
    // 64 lanes of a load fill 1 KB of consecutive LDS, which rules out padded rows).  A tile of 32
    // rows is kept as [k-step ks][row][64 bytes]: the 4 chunks of 16 bytes that a row holds of
    // head-dim columns 32 ks .. 32 ks + 31, chunk c at position c ^ s(row) with s = row / 4 mod 4 for
    // K and the same two bits swapped for V.  The row fragments of K (lane n reads row n) and the
    // transposed fragments of V then touch every bank equally often, and k-step, row block and head-dim
    // block are constant offsets from one lane address.
    static constexpr int KST = D * 2;              // bytes of a row in global memory
    static constexpr int k_bytes = BK * KST;
    static constexpr int buf_bytes = 2 * k_bytes;  // K rows, then V rows
    // two buffers: the rows of step u+1 arrive during step u (3 or 4, two or three steps ahead, measured no faster, with one
    // workgroup per CU neither)
    static constexpr int total = 2 * buf_bytes;
};

// A query tile's key steps cut into parts of at most `share` steps, one workgroup each (0: one workgroup per tile); a part
// leaves its O (not normalised), row sums, exponent bases and maxima in `part`, [batch, head][workgroup][BQ][D + 4] fp32, for
// fwd_merge_kernel.
struct FwdSplit { int share, first_long; float *part; };
template <int BQ>
__host__ __device__ inline int fwd_steps(const Problem &p, int qt) {
    const int k_end = p.causal ? (p.Nk < (qt + 1) * BQ ? p.Nk : (qt + 1) * BQ) : p.Nk;
    return (k_end + 16 + BK - 1) / BK;
}
__host__ __device__ inline int fwd_parts(int steps, int share) { return share > 0 && steps > share ? (steps + share - 1) / share : 1; }
template <int BQ> inline int fwd_wgs(const Problem &p, int share) {
    int n = 0;
    for (int qt = 0; qt < (p.Nq + BQ - 1) / BQ; ++qt) n += fwd_parts(fwd_steps<BQ>(p, qt), share);
    return n;
}

// Waves per SIMD that the registers have to leave room for: windows of up to 6 slots fit three (168 registers) up to d = 64.  Forced to
// three, 7 and 8 slots spill (B4 H16 N4096 d64 7x7 324 -> 402 us, 8x11 340 -> 380, B2 H12 N3000 7x7 79 -> 109); four at d = 32 with 3 slots:
// the same (B4 H16 N4096 154 and 156).
constexpr int fwd_waves(int d, int cqt) { return d <= 64 && cqt <= 6 ? 3 : 2; }
// (SPLIT: an instance of its own, the other one is a percent slower with the parts' bounds at run time)
// LONG: the tiles from split.first_long on run at a higher wave priority (long_tiles_first)
enum { PLAIN, SPLIT_KEYS, LONG };
// WIDE: windows of 17 key taps, whose band the sparse product cannot hold (each tap a dense product of its own)
template <int D, int CQT, typename TO, int FORM, bool WIDE>
__global__ __launch_bounds__(NW * 64, fwd_waves(D, CQT)) void fwd_reg_mfma_kernel(
    Problem p, FwdSplit split, const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K,
    const bf16_t *__restrict__ V, const float *__restrict__ W, TO *__restrict__ O,
    float *__restrict__ M, float *__restrict__ L) {
    using Lds = FwdLds<D>;
    constexpr bool SPLIT = FORM == SPLIT_KEYS;
    constexpr int KST = Lds::KST;
    constexpr int KS = D / 32;   // MFMA k-steps over the head dimension
    constexpr int DB = D / 16;   // 16-wide blocks of the head dimension
    constexpr int WR = wave_rows(CQT), BQ = NW * WR;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;  // wave-uniform for the compiler too
    const int g = lane >> 4, n = lane & 15;

    // x = head, y = batch, z = query tile: the dispatcher hands out every (batch, head) of the
    // longest (causal) tiles first, so the tail of the launch is made of short tiles
    const int h = blockIdx.x, b = blockIdx.y;
    int qt = gridDim.z - 1 - blockIdx.z, part_no = 0;
    if constexpr (SPLIT)
        for (qt = (p.Nq + BQ - 1) / BQ - 1, part_no = blockIdx.z; part_no >= fwd_parts(fwd_steps<BQ>(p, qt), split.share); --qt)
            part_no -= fwd_parts(fwd_steps<BQ>(p, qt), split.share);
    const int i0 = qt * BQ, i0w = i0 + wave * WR;
    const bool is_long = FORM == LONG && qt >= split.first_long;
    if (is_long) __builtin_amdgcn_s_setprio(3);
    const int base = i0w - (CQT - 1);  // first score row of the wave
    const int pk = p.pk, cq = p.c_q;
    const bool causal = p.causal != 0;
    const size_t bh = (size_t)b * p.H + h;
    const bf16_t *Qb = Q + bh * p.Nq * D;
    const bf16_t *Kb = K + bh * p.Nk * D;
    const bf16_t *Vb = V + bh * p.Nk * D;

    const int all_steps = fwd_steps<BQ>(p, qt), parts = SPLIT ? fwd_parts(all_steps, split.share) : 1;
    const int u_lo = SPLIT ? all_steps * part_no / parts : 0, n_steps = SPLIT ? all_steps * (part_no + 1) / parts : all_steps;   // this workgroup's steps
    // (a part that does not begin with the first step takes the scores of the step before it along the way: the window
    // needs the last block of them)
    const int u_first = SPLIT ? max(u_lo - 1, 0) : 0;

    // Toeplitz bands of this head, pre-multiplied by scale * log2(e): the convolved scores come out in log2 units.  WIDE: k slot
    // 8g+e of a window is key 4g+e of its first 16-key block for e < 4, key 4g+e-4 of its second for e >= 4.
    using Taps = SparseTaps<CQT>;
    f16x8 tf[WIDE ? CQT : 1];
    SparseBands<CQT, (CQT <= 7 || D <= 64)> bands;   // (11 slots at d = 128 have no registers for both orders of the single slots' blocks)
    int index[2] = {0, 0};   // of the windows that end with a step's first and second score block
    {
        // (the table lies in the K / V buffer that the first step does not use)
        static_assert(band_table_bytes<CQT>() <= Lds::buf_bytes, "room for the table");
        unsigned int *tab = reinterpret_cast<unsigned int *>(smem + ((u_first & 1) ^ 1) * Lds::buf_bytes);
        band_table_build<CQT>(tab, W + (size_t)h * cq * p.c_k, cq, p.c_k, pk, p.scale * kLog2e, tid, NW * 64);
        __syncthreads();
        if constexpr (WIDE) {
#pragma unroll
            for (int t = 0; t < CQT; ++t) {
                u32x4 v;
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = tab[t * kBandRow + 4 * g + 2 * (q & 1) + (q >> 1) * 16 - n + 16];
                tf[t] = __builtin_bit_cast(f16x8, v);
            }
        } else {
            bands.read(tab, g, n);
            index[0] = sparse_index(g, n, true);
            index[1] = sparse_index(g, n, false);
        }
    }

    // Q^T fragments (B operand), resident for the whole loop: lane n of fragment f holds row
    // base + 2n + f, so a shift of the score rows by an even number of rows is a shift of
    // lanes and by an odd number a change of fragment as well.
    bf16x8 qf[2][KS];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            qf[f][ks] = __builtin_bit_cast(bf16x8, load_row16_nb<D>(Qb, base + 2 * n + f, p.Nq, ks * 32 + g * 8));

    f32x4 acc_o[2][DB];
#pragma unroll
    for (int ob = 0; ob < 2; ++ob)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc_o[ob][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m_ref[2] = {kNegInf, kNegInf};   // exponent base of the row, in log2 units (same in the row's 4 lanes)
    float m_rel[2] = {kNegInf, kNegInf};   // maximum of the scores this lane has seen, relative to m_ref (or 0)
    // The convolution accumulates on top of minus the exponent base (0 while the row has none),
    // so its result is already the exponent; slack[ob]: how far it may go above 0 before the base
    // is raised (-inf while the row has no base: any visible score sets one).
    f32x4 neg_base[2] = {(f32x4){0.f, 0.f, 0.f, 0.f}, (f32x4){0.f, 0.f, 0.f, 0.f}};
    float slack[2] = {kNegInf, kNegInf};
    float l_run[2] = {0.f, 0.f};           // this lane's share of the row sum, relative to m_ref

    // Step u: score blocks 2u, 2u+1 (keys 32u-8 .. 32u+23, K rows of the step) and output blocks
    // 2u-1, 2u (keys 32u-16 .. 32u+15, V rows of the step); an output block needs the score
    // block 8 keys before it and the one 8 keys after it, so the packed scores of block 2u-1
    // are carried from the previous step.
    // K / V rows: buffer loads with the LDS modifier.  Rows before the first or after the last key
    // are outside the descriptor's range and arrive as zeros, which is what the window's zero
    // padding asks for.
    // A tile is 2 KS units of 1 KB (unit 2 ks + blk = rows 16 blk .. 16 blk + 15 of k-step ks); wave w
    // issues the units w, w + NW, ...  Lane l of a load fills chunk position l % 4 of row l / 4.
    // (head dimension 32: two units, issued by the waves 0 and 1)
    constexpr int UNITS = Lds::k_bytes / 1024, N_LD = UNITS >= NW ? UNITS / NW : 1;
    static_assert(UNITS == 2 * KS && (UNITS % NW == 0 || UNITS < NW) && NW == 4, "whole units per wave");
    const bool dma_wave = UNITS >= NW || wave < UNITS;
    // (K rows are read as row fragments, 16 rows of one chunk column at a time: swizzle value row / 4 mod 4;
    // V rows through transpose reads, 8 rows x 32 bytes per half wave: the same value with its two bits
    // swapped, so that rows r and r + 4 use different halves of their 64 bytes)
    const int dma_row = (16 * (wave & 1) + (lane >> 2)) * KST;
    const int dma_off = dma_row + (((wave >> 1) * 4 + ((lane & 3) ^ ((lane >> 4) & 3))) << 4);
    const int dma_off_v = dma_row + (((wave >> 1) * 4 + ((lane & 3) ^ ((((lane >> 4) & 1) << 1) | ((lane >> 5) & 1)))) << 4);
    // rows of step u: issued right after the barrier that ends step u - 1 (their buffer is free then),
    // landed by the barrier that starts step u (the barrier waits for the wave's loads)
    // (issued as inline assembly: for the builtin the compiler makes every later LDS read wait for the
    // load, since it cannot tell the two buffers apart; the wait is written out before the barrier instead)
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    auto dma_rsrc = [&](const bf16_t *ptr) {
        const unsigned long long a = reinterpret_cast<unsigned long long>(ptr);
        return (i32x4){(int)(unsigned int)a, (int)(unsigned int)(a >> 32), p.Nk * D * 2, 0x00020000};
    };
    const i32x4 k_dma = dma_rsrc(Kb), v_dma = dma_rsrc(Vb);
    const unsigned int lds_u = (unsigned int)(unsigned long long)(__attribute__((address_space(3))) unsigned char *)smem;
    const unsigned int lds_base = lds_u + wave * 1024;
    // unit i of the wave: k-step + 2 i = 128 bytes further along the row (the instruction's offset
    // field, which the hardware adds to the LDS address as well as to the global one), 4 KB further in
    // LDS; the step's first row is the scalar offset of the load
    auto dma16 = [&](const i32x4 &rsrc, unsigned int lds_addr, int voffset, int soffset, auto I) {
        constexpr int i = decltype(I)::value;
        // (M0 is written here and read by the load that follows; nothing else of this kernel uses it)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen offset:%4 lds"
                     :: "s"(__builtin_amdgcn_readfirstlane((int)lds_addr + i * (4096 - 128))), "v"(voffset), "s"(rsrc),
                        "s"(__builtin_amdgcn_readfirstlane(soffset)), "n"(i * 128) : "memory");
    };
    // step 0 starts before the first key: those rows have negative offsets, which only the vector
    // offset (a wrapping 32-bit sum made here) may carry; later steps pass theirs as the scalar offset
    auto fetch_step = [&](int u) {
        const unsigned int Ks = lds_base + (u & 1) * Lds::buf_bytes, Vs = Ks + Lds::k_bytes;
        const int k0 = (32 * u - 8) * KST, v0 = (32 * u - 16) * KST;
        if (dma_wave) static_for<N_LD>([&](auto I) {
            if (u == 0) {
                dma16(k_dma, Ks, dma_off + k0, 0, I);
                dma16(v_dma, Vs, dma_off_v + v0, 0, I);
            } else {
                // (a scalar offset past the end is held at the end: everything is out of range then,
                // whichever way the range check treats a scalar offset beyond the number of records)
                dma16(k_dma, Ks, dma_off, min(k0, p.Nk * KST), I);
                dma16(v_dma, Vs, dma_off_v, min(v0, p.Nk * KST), I);
            }
        });
    };
    // lane addresses (absolute LDS addresses) of the fragment reads inside the buffer of the step; they
    // are moved to the other buffer at the end of every step.  K row fragment: row n, chunk 4 ks + g;
    // row block and k-step are constant offsets.  V^T fragment: rows 4g + n/4 (+ 16), 8 bytes at byte
    // column 32 db + 8 (n % 4): head-dim blocks 2 x and 2 x + 1 differ in bit 5 of the lane part.
    unsigned int ka = opaque_u32(lds_u + n * 64 + ((g ^ ((n >> 2) & 3)) << 4));
    unsigned int va[2];
    va[0] = opaque_u32(lds_u + Lds::k_bytes + (4 * g + (n >> 2)) * 64 + ((((n >> 1) & 1) ^ (((g & 1) << 1) | (g >> 1))) << 4) + (n & 1) * 8);
    va[1] = opaque_u32(va[0] ^ 32u);
    typedef __attribute__((address_space(3))) const bf16x8 *lds_bf16x8_ptr;
    typedef __attribute__((address_space(3))) const unsigned char *lds_byte_ptr;

    // packed fp16 scores of the last score block of the previous step:
    // carry[f][dword] = row base + 2n + f, keys 4g .. 4g+3 of the block
    unsigned int carry[2][2] = {{0u, 0u}, {0u, 0u}};
    // The sparse products' operands, kept from step to step: a step's first score block has the even dwords of the tuples, its
    // second one the odd ones, and each takes the place of the block two before it.  Every row offset of a block is made once
    // (CQT - 1 DPP moves of two dwords) and serves the two windows the block is in.
    u32x8 rows[WIDE ? 1 : Taps::tuples];
    if constexpr (!WIDE)
#pragma unroll
        for (int j = 0; j < Taps::tuples; ++j) rows[j] = (u32x8)0u;
    // dwords of tuple j from the packed scores pd[f][dword] of a block
    auto put_rows = [&](auto J, auto BLK, const unsigned int (&pd)[2][2]) {
        constexpr int j = decltype(J)::value, blk = decltype(BLK)::value;
        static_for<2>([&](auto HALF) {
            constexpr int half = decltype(HALF)::value, delta = Taps::delta(j, half), f = delta & 1, s = (f - delta) / 2;
#pragma unroll
            for (int dw = 0; dw < 2; ++dw) {
                if constexpr (s == 0) rows[j][4 * half + 2 * dw + blk] = pd[f][dw];
                else rows[j][4 * half + 2 * dw + blk] = dpp_zero<0x110 + s>(pd[f][dw]);
            }
        });
    };

    // One step of the wave; EDGE = the step touches the diagonal or an end of the keys
    // (wave-uniform), only then are the masks evaluated.
    auto step = [&](int u, auto edge_tag) {
        constexpr bool EDGE = decltype(edge_tag)::value;
        const int jk = 32 * u - 8, jv = 32 * u - 16;
        f32x4 c[2][2];
        bf16x8 kf[KS];  // K fragments of one score block; the second block's are read during the first's convolution
        unsigned int pd[2][2][2];  // [score block of the step][f][dword]
        auto load_kf = [&](int blk) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                kf[ks] = *(lds_bf16x8_ptr)(size_t)(ka + blk * 1024 + ks * 2048);
        };
        load_kf(0);
        static_for<2>([&](auto BL) {
            constexpr int blk = decltype(BL)::value;
            // ---- S^T = K Q^T (raw), pre-mask, pack two keys per dword ----
            f32x4 acc[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) acc[f] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int f = 0; f < 2; ++f) acc[f] = mfma_bf16(kf[ks], qf[f][ks], acc[f]);
            if constexpr (blk == 0) {
                load_kf(1);
                SCHED_DS_READ(KS);
                SCHED_MFMA(WIDE ? 2 * CQT : 2 * (Taps::products + Taps::odd));
            }
            const int key0 = jk + blk * 16 + 4 * g;
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                if constexpr (EDGE) {
                    if (causal) {
                        const int qpos = base + 2 * n + f;
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (key0 + r > qpos) acc[f][r] = 0.f;
                    }
                }
                const u32x2 two = pack_scores_f16(acc[f]);
                pd[blk][f][0] = two[0];
                pd[blk][f][1] = two[1];
            }
            // ---- convolution of output block blk: one B operand per row offset
            //      delta = (output row parity) + (tap slot) - (CQT-1): rows base + 2n + delta =
            //      fragment f shifted s lanes down (zeros shifted in: those lanes are halo rows,
            //      whose outputs are not used); k slots 0..3 of a lane group from the score block
            //      before, 4..7 from this one ----
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) c[ob][blk] = neg_base[ob];
            if constexpr (!WIDE) {
                auto single = [&](auto OB) {   // (the first product of its parity, which brings the chain's starting value with it)
                    constexpr int ob = decltype(OB)::value;
                    c[ob][blk] = bands.single(1 - blk, ob, rows[Taps::single_tuple(ob)], c[ob][blk]);
                };
                if constexpr (Taps::odd) {
                    put_rows(std::integral_constant<int, Taps::tuples - 1>{}, BL, pd[blk]);
                    single(std::integral_constant<int, 0>{});
                }
                static_for<Taps::tuples>([&](auto J) {
                    constexpr int j = decltype(J)::value;
                    if constexpr (!Taps::odd || j < Taps::tuples - 1) put_rows(J, BL, pd[blk]);
                    if constexpr (Taps::odd && j == 0) single(std::integral_constant<int, 1>{});
                    static_for<2>([&](auto OB) {
                        constexpr int ob = decltype(OB)::value;
                        static_for<Taps::products>([&](auto I) {
                            constexpr int i = decltype(I)::value;
                            if constexpr (Taps::tuple(i, ob) == j) c[ob][blk] = smfmac_f16(bands.band[ob][i], rows[j], c[ob][blk], index[blk]);
                        });
                    });
                });
            }
            else static_for<CQT + 1>([&](auto DL) {
                constexpr int delta = decltype(DL)::value - (CQT - 1);
                constexpr int f = delta & 1, s = (f - delta) / 2;
                u32x4 bv;
#pragma unroll
                for (int half = 0; half < 2; ++half)
#pragma unroll
                    for (int dw = 0; dw < 2; ++dw) {
                        const unsigned int own = half ? pd[blk][f][dw] : (blk ? pd[0][f][dw] : carry[f][dw]);
                        if constexpr (s == 0) bv[2 * half + dw] = own;
                        else bv[2 * half + dw] = dpp_zero<0x110 + s>(own);
                    }
                constexpr int t0 = delta + (CQT - 1);  // tap slot of output parity 0
                if constexpr (t0 < CQT) c[0][blk] = mfma_f16(tf[t0], __builtin_bit_cast(f16x8, bv), c[0][blk]);
                if constexpr (t0 >= 1) c[1][blk] = mfma_f16(tf[t0 - 1], __builtin_bit_cast(f16x8, bv), c[1][blk]);
            });
        });
        if constexpr (WIDE)
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int dw = 0; dw < 2; ++dw) carry[f][dw] = pd[1][f][dw];
        // V^T fragments of the first kFwdPfv head-dim blocks: in flight during the softmax
        constexpr int PFV = kFwdPfv < DB ? kFwdPfv : DB;
        bf16x8 vf[PFV + 1];
        auto load_vf = [&](int buf, int db) {
            bf16x4 lo = lds_tr64((lds_byte_ptr)(size_t)(va[db & 1] + (db >> 1) * 2048));
            bf16x4 hi = lds_tr64((lds_byte_ptr)(size_t)(va[db & 1] + (db >> 1) * 2048 + 1024));
            vf[buf] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
#pragma unroll
        for (int db = 0; db < PFV; ++db) load_vf(db, db);
        // The two waves of a SIMD are at different places of their steps: the one in an MFMA
        // phase (P V, S^T, the convolution) gets the issue slot first, the one in the softmax
        // arithmetic fills the gaps (measured: 1.5 % over equal priorities; the reverse is slower).
        if (!is_long) __builtin_amdgcn_s_setprio(0);
        // ---- post-mask and softmax numerators (log2 domain).  The exponent base m_ref of a row
        //      only follows the row's maximum when some score exceeds it by more than kMaxSlack
        //      (then every lane group of the wave exchanges its maxima and rescales); otherwise no
        //      lane talks to another.  The true maximum is tracked per lane for the M output. ----
#pragma unroll
        for (int ob = 0; ob < 2; ++ob) {
            if constexpr (EDGE) {
                const int qpos = base + 2 * n + ob;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int key = jv + kb * 16 + 4 * g + r;
                        if (key < 0 || key >= p.Nk || (causal && key > qpos)) c[ob][kb][r] = kNegInf;
                    }
            }
            // (the maximum so far never lies above the slack, so the test below may include it)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) m_rel[ob] = fmaxf(m_rel[ob], c[ob][kb][r]);
        }
        if (__builtin_amdgcn_ballot_w64(m_rel[0] > slack[0] || m_rel[1] > slack[1]) != 0) {
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) {
                const float old_use = -neg_base[ob][0];
                float mx = m_rel[ob] + old_use;
                mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
                mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
                const float m_new = fmaxf(m_ref[ob], mx);
                // rows with nothing visible yet keep m = -inf; 0 is the exponent base there
                const float new_use = (m_new == kNegInf) ? 0.f : m_new;
                const float alpha = fast_exp2(m_ref[ob] - new_use);
                const float delta = new_use - old_use;
                m_ref[ob] = m_new;
                if (new_use < -kNegInf) m_rel[ob] -= delta;   // (under a base of +inf it stays +inf: inf - inf is no maximum)
                slack[ob] = (m_new == kNegInf) ? kNegInf : kMaxSlack;
                neg_base[ob] = (f32x4){-new_use, -new_use, -new_use, -new_use};
                l_run[ob] *= alpha;
#pragma unroll
                for (int db = 0; db < DB; ++db) acc_o[ob][db] *= alpha;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) c[ob][kb][r] -= delta;
            }
        }
#pragma unroll
        for (int ob = 0; ob < 2; ++ob) {
            float psum = 0.f;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float e = fast_exp2(c[ob][kb][r]);
                    c[ob][kb][r] = e;
                    psum += e;
                }
            l_run[ob] += psum;
        }
        // ---- O^T += V^T P^T: V^T fragments through the LDS transpose read, P^T straight from
        //      the softmax registers (k slot 8g+e <-> key 4g+e of output block 0 for e < 4, of
        //      output block 1 for e >= 4) ----
        if (!is_long) __builtin_amdgcn_s_setprio(1);
        bf16x8 pf[2];
#pragma unroll
        for (int ob = 0; ob < 2; ++ob)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pf[ob][r] = (bf16_t)c[ob][0][r];
                pf[ob][4 + r] = (bf16_t)c[ob][1][r];
            }
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (db + PFV < DB) {
                load_vf((db + PFV) % (PFV + 1), db + PFV);
                SCHED_DS_READ(2);
            }
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) acc_o[ob][db] = mfma_bf16(vf[db % (PFV + 1)], pf[ob], acc_o[ob][db]);
            SCHED_MFMA(2);
        }
    };

    fetch_step(u_first);
    if constexpr (SPLIT) {
        const int to_first = (u_first & 1) * Lds::buf_bytes;
        ka += to_first;
        va[0] += to_first;
        va[1] += to_first;
    }
    auto carry_only = [&](int u) {
        const int jk = 32 * u + 8;   // keys of the step's second block
        f32x4 acc[2] = {(f32x4){0.f, 0.f, 0.f, 0.f}, (f32x4){0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int f = 0; f < 2; ++f)
                acc[f] = mfma_bf16(*(lds_bf16x8_ptr)(size_t)(ka + 1024 + ks * 2048), qf[f][ks], acc[f]);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const int qpos = base + 2 * n + f;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (causal && jk + 4 * g + r > qpos) acc[f][r] = 0.f;
            const u32x2 two = pack_scores_f16(acc[f]);
            carry[f][0] = two[0];
            carry[f][1] = two[1];
        }
        if constexpr (!WIDE) static_for<Taps::tuples>([&](auto J) { put_rows(J, std::integral_constant<int, 1>{}, carry); });
    };
    // Along the keys a wave's steps are: step 0 (keys before the first one to mask), steps whose
    // keys all lie at or before its first score row (no masks), steps on the diagonal or at the
    // end of the keys (masks), and steps entirely after its rows (it only takes part in the
    // staging).  One loop per kind, so that each loop body has the accumulators in place.
    auto run = [&](int ua, int ub, auto kind) {
        constexpr int KIND = decltype(kind)::value;
#pragma unroll 1
        for (int u = ua; u < ub; ++u) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's rows of step u have landed
            __syncthreads();  // step u-1 is done everywhere: its buffer is free, and step u's is written
            if (!SPLIT || u + 1 < n_steps) fetch_step(u + 1);
            if constexpr (KIND == 3) carry_only(u);
            else if constexpr (KIND != 2) step(u, std::integral_constant<bool, KIND == 1>{});
            const int to_other = (u & 1) ? -Lds::buf_bytes : Lds::buf_bytes;
            ka += to_other;
            va[0] += to_other;
            va[1] += to_other;
        }
    };
    const int u_diag = base < 23 ? 1 : (base - 23) / 32 + 1;    // first u >= 1 with 32u + 23 > base
    const int u_tail = p.Nk < 24 ? 1 : (p.Nk - 24) / 32 + 1;    // first u >= 1 with 32u + 24 > Nk
    const int u1 = min(causal ? min(u_diag, u_tail) : u_tail, n_steps);
    const int u2 = max(u1, causal ? min((i0w + WR + 15) / 32 + 1, n_steps) : n_steps);  // 32u - 16 > i0w + WR - 1
    if constexpr (SPLIT) run(u_first, u_lo, std::integral_constant<int, 3>{});
    run(u_lo, 1, std::integral_constant<int, 1>{});
    run(max(1, u_lo), u1, std::integral_constant<int, 0>{});
    run(max(u1, u_lo), u2, std::integral_constant<int, 1>{});
    run(max(u2, u_lo), n_steps, std::integral_constant<int, 2>{});
    // ---- epilogue: finish the row sums and maxima, normalise, store O, M, L ----
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
        float l = l_run[ob];
        l += __shfl_xor(l, 16, kWave);
        l += __shfl_xor(l, 32, kWave);
        float mt = m_rel[ob] - neg_base[ob][0];
        mt = fmaxf(mt, __shfl_xor(mt, 16, kWave));
        mt = fmaxf(mt, __shfl_xor(mt, 32, kWave));
        const int qpos = base + 2 * n + ob;
        if (SPLIT && parts > 1) {
            if (qpos >= i0w && qpos < p.Nq) {
                float *dst = split.part + ((bh * gridDim.z + blockIdx.z) * BQ + qpos - i0) * (D + 4);
#pragma unroll
                for (int db = 0; db < DB; ++db) *reinterpret_cast<f32x4 *>(dst + db * 16 + 4 * g) = acc_o[ob][db];
                if (g == 0) *reinterpret_cast<f32x4 *>(dst + D) = (f32x4){l, m_ref[ob], mt, 0.f};
            }
            continue;
        }
        if (qpos >= i0w && qpos < p.Nq) {
            const float inv = 1.f / l;
            TO *orow = O + (bh * p.Nq + qpos) * D;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const int col = db * 16 + 4 * g;
                if constexpr (sizeof(TO) == 2) {
                    bf16x4 ov;
#pragma unroll
                    for (int r = 0; r < 4; ++r) ov[r] = (bf16_t)(acc_o[ob][db][r] * inv);
                    *reinterpret_cast<bf16x4 *>(orow + col) = ov;
                } else {
                    f32x4 ov = acc_o[ob][db] * inv;
                    *reinterpret_cast<f32x4 *>(orow + col) = ov;
                }
            }
            if (g == 0) {
                M[bh * p.Nq + qpos] = mt * (1.f / kLog2e);
                L[bh * p.Nq + qpos] = l * fast_exp2(m_ref[ob] - mt);
            }
        }
    }
}

// O, M and L of the rows of a split query tile from its parts: 4 columns of a row per thread.
// x = 256 threads of the tile, y = tile from the last on, z = (batch, head).
template <int D, int BQ, typename TO>
__global__ __launch_bounds__(256) void fwd_merge_kernel(Problem p, FwdSplit split, int n_wg, TO *__restrict__ O, float *__restrict__ M,
                                                        float *__restrict__ L) {
    int z = 0, qt = (p.Nq + BQ - 1) / BQ - 1;
    for (int i = 0; i < (int)blockIdx.y; ++i, --qt) z += fwd_parts(fwd_steps<BQ>(p, qt), split.share);
    const int parts = fwd_parts(fwd_steps<BQ>(p, qt), split.share);
    const int e = blockIdx.x * 256 + threadIdx.x, r = e / (D / 4), col = (e % (D / 4)) * 4, row = qt * BQ + r;
    if (r >= BQ || row >= p.Nq) return;
    const float *src = split.part + (((size_t)blockIdx.z * n_wg + z) * BQ + r) * (D + 4);
    const size_t step = (size_t)BQ * (D + 4);
    float ref = kNegInf, m = kNegInf, l = 0.f;
    for (int i = 0; i < parts; ++i) {
        const f32x4 st = *reinterpret_cast<const f32x4 *>(src + i * step + D);
        ref = fmaxf(ref, st[1]);
        m = fmaxf(m, st[2]);
    }
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < parts; ++i) {   // (a part none of whose keys the row sees has base -inf: factor 0)
        const f32x4 st = *reinterpret_cast<const f32x4 *>(src + i * step + D);
        const float f = fast_exp2(st[1] - ref);
        l = fmaf(st[0], f, l);
        o += *reinterpret_cast<const f32x4 *>(src + i * step + col) * f;
    }
    o *= 1.f / l;
    const size_t at = (size_t)blockIdx.z * p.Nq + row;
    if constexpr (sizeof(TO) == 2) {
        const bf16x4 ov = {(bf16_t)o[0], (bf16_t)o[1], (bf16_t)o[2], (bf16_t)o[3]};
        *reinterpret_cast<bf16x4 *>(O + at * D + col) = ov;
    } else {
        *reinterpret_cast<f32x4 *>(O + at * D + col) = o;
    }
    if (col == 0) {
        M[at] = m * (1.f / kLog2e);
        L[at] = l * fast_exp2(ref - m);
    }
}

// Steps per workgroup, or 0: one workgroup per query tile.  In units of a key step of a workgroup that has a CU to itself:
// a workgroup costs its steps and about 4 (5 where it is a part); with two per CU each runs at 0.6 of that; the merge
// kernel about 8.  Few (batch, head) pairs or rows leave the launch as long as its longest tile
// (B1 H8 N2048 d64 7x7: 41 -> 34 us with the merge, B1 H8 N1000 d128 6x11: 28 -> 25).
// What this leaves out is the traffic of the parts, D + 4 floats per row and part: with many unsplit workgroups for their length
// the split form is slower (B2 H16 N2048 6x11: d64 54 us unsplit, 60 in parts, d128 69 and 87; 3x3 d128 61 and 81), so it is
// taken up to `fill` of them only.  The line was drawn with one dense product per tap: of 753 shapes of 1 to 64 heads and 1000 to 8000
// rows (3x3 to 11x11 taps, d 32 to 128) that the estimate splits, 6 were up to 4 % slower than unsplit with it (105, up to 38 %, without).
// With the present steps, 11 to 23 % shorter, of 150 other such shapes 73 run in parts, in 0.75 of the unsplit time on average, 12 of them
// 3 to 8 % slower than unsplit; 7 unsplit ones would gain more than 3 %.  The cut taken is 2.8 % over the best of up to six parts on
// average (unsplit: 25 %), single ones up to 27 % (B1 H2 N7781 d128 8x15 109 us, in five parts 86).
// Sequences of less than 32 steps would gain too (B1 H8 N640 d64 6x11 16.0 -> 15.1 us); their calls are bound by the host.  Beyond 64
// heads no cut gained (13 to 55 % slower at 80 to 256 heads of 1024 to 4096 rows, dense products).  From 8192 rows on nothing is split, whatever
// the number of heads is, so that a head's results do not depend on how many others there are; up to four heads would gain
// (B1 H1 N16384 d128 349 -> 156 us, B1 H4 N8192 190 -> 152), more would not (B1 H8 N8192 237 -> 259).
template <int BQ> int fwd_share(const Problem &p) {
    const int n_qt = (p.Nq + BQ - 1) / BQ, most = fwd_steps<BQ>(p, n_qt - 1);
    if (most < 32 || p.Nq >= 8192 || p.Nk >= 8192 || p.B * (long long)p.H > 64) return 0;
    float none = 0.f, best = 0.f;
    int share = 0;
    for (int cut = 1; cut <= 6; ++cut) {
        const int sh = cut == 1 ? 0 : (most + cut - 1) / cut;
        if (cut > 1 && sh < 6) break;
        float total = 0.f, longest = 0.f;
        int jobs = 0;
        for (int qt = 0; qt < n_qt; ++qt) {
            const int st = fwd_steps<BQ>(p, qt), parts = fwd_parts(st, sh);
            const float one = (float)((st + parts - 1) / parts) + (parts > 1 ? 5.f : 4.f);
            longest = one > longest ? one : longest;
            total += one * parts;
            jobs += parts;
        }
        const float n = (float)p.B * p.H, even = total * n / (256.f * 1.22f) + 0.35f * longest;
        const float alone = jobs * n <= 256.f ? longest : jobs * n >= 512.f ? 1.64f * longest : (1.f + 0.64f * (jobs * n - 256.f) / 256.f) * longest;
        const float t = jobs * n <= 256.f || alone > even ? alone : even;
        if (cut == 1) {
            const float fill = 205.f + most * (p.d <= 64 ? 1.7f : p.c_q <= 6 ? 1.25f : 1.4f);
            // (not causal: one full round of equal workgroups; 3 query taps: the shortest steps)
            if (jobs * n > fill || (!p.causal && jobs * n > 200.f && jobs * n <= 256.f) || (p.c_q <= 3 && most < 36 && jobs * n > 100.f))
                return 0;
            none = best = t;
        } else if (1.1f * t + 8.f < none && t < best) { best = t; share = sh; }
    }
    return share;
}

// Causal launches of 1.4 to 2 rounds of workgroups end with their longest tiles: a CU has three workgroups, a slot's tiles are shorter
// together than the longest one alone (65 and 55 steps at B4 H16 N2048 d64 6x11), and that one runs at a third of the CU until the others
// leave.  There the longer half of the tiles gets the issue slots first; us without and with it at B4 H16 N2048 (1.6 rounds): d64 6x11
// 86 / 80, 3x3 70 / 65, d32 6x11 66 / 63.
// Below 1.4 and beyond 2 rounds the two waves of a SIMD had better take turns by phase (d64): 6x11 of 1.17 rounds (32 heads) 82.6 / 85.1, d32 of 1.41
// (24 heads) 115 / 122; 2.17 130 / 131, 2.4 397 / 399, B4 H16 N4096 (3.2) 264 / 269.
// The fewer tiles a head has, the less there is to put in order, and the earlier that ends: with 47 tiles (B1 H32 N5000) 1.96 rounds 213 / 204, 22
// tiles 1.83 rounds 101 / 96; 10 tiles 1.67 rounds 49.5 / 48.2.  That end was drawn with one dense product per tap (144 launches of 64 to 384 heads;
// 24 tiles (B4 H16 N2581) 2.0 rounds 137 / 144, 7 tiles (B12 H16 N745) 1.75 48.4 / 49.0); now these would gain as well (118 / 112, 41.9 / 40.0), and so
// would 7 and 8 slots at d = 32, which have three workgroups per CU since (B4 H16 N2048 7x7 71 / 65, 8x15 80 / 74).
// The instances that had three workgroups per CU then; with two it costs up to 10 % in this band (B1 H32 N2500 d64 7x7 64 / 71), with four (d32 3x3)
// 1 to 4 %.
constexpr bool has_long(int d, int cqt) { return (d == 64 && cqt <= 6) || (d == 32 && cqt == 6); }
template <int BQ> bool long_tiles_first(const Problem &p) {
    const long long tiles = (p.Nq + BQ - 1) / BQ, wgs = p.B * p.H * tiles, round = 3 * 256;
    return p.causal && 5 * wgs > 7 * round && wgs <= 2 * round && 10 * wgs * tiles <= (21 * tiles - 30) * round;   // (up to 2.1 - 3 / tiles rounds)
}

template <int D, int CQT, typename TO, bool WIDE>
hipError_t launch_fwd(const Problem &p, float *part, const void *q, const void *k, const void *v, const float *w,
                      void *o, float *m, float *l, hipStream_t s) {
    constexpr int lds = FwdLds<D>::total, BQ = NW * wave_rows(CQT);
    if (lds > 64 * 1024) {
        hipError_t e = set_max_lds_once<fwd_reg_mfma_kernel<D, CQT, TO, PLAIN, WIDE>>(lds);
        if (e == hipSuccess) e = set_max_lds_once<fwd_reg_mfma_kernel<D, CQT, TO, SPLIT_KEYS, WIDE>>(lds);
        if (e != hipSuccess) return e;
    }
    const FwdSplit split{part ? fwd_share<BQ>(p) : 0, (p.Nq + BQ - 1) / BQ / 2, part};
    const int n_wg = fwd_wgs<BQ>(p, split.share);
    auto kern = split.share ? fwd_reg_mfma_kernel<D, CQT, TO, SPLIT_KEYS, WIDE> : fwd_reg_mfma_kernel<D, CQT, TO, PLAIN, WIDE>;
    if constexpr (has_long(D, CQT))
        if (!split.share && long_tiles_first<BQ>(p)) kern = fwd_reg_mfma_kernel<D, CQT, TO, LONG, WIDE>;
    kern<<<dim3(p.H, p.B, n_wg), NW * 64, lds, s>>>(p, split, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, w, (TO *)o, m, l);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !split.share) return e;
    int tiles = 0;   // (the split tiles are the last ones)
    const int n_qt = (p.Nq + BQ - 1) / BQ;
    while (tiles < n_qt && fwd_parts(fwd_steps<BQ>(p, n_qt - 1 - tiles), split.share) > 1) ++tiles;
    fwd_merge_kernel<D, BQ, TO><<<dim3((BQ * D / 4 + 255) / 256, tiles, p.B * p.H), 256, 0, s>>>(p, split, n_wg, (TO *)o, m, l);
    return hipGetLastError();
}

template <int D, typename TO, bool WIDE>
hipError_t pick_cq(const Problem &p, float *part, const void *q, const void *k, const void *v, const float *w,
                   void *o, float *m, float *l, hipStream_t s) {
    if (p.c_q <= 3) return launch_fwd<D, 3, TO, WIDE>(p, part, q, k, v, w, o, m, l, s);
    if (p.c_q <= 6) return launch_fwd<D, 6, TO, WIDE>(p, part, q, k, v, w, o, m, l, s);
    // (7 taps in 8 slots, B2 H12 N4691: d128 231 us, in 7 225, d64 170 and 157)
    if (p.c_q <= 7) return launch_fwd<D, 7, TO, WIDE>(p, part, q, k, v, w, o, m, l, s);
    if (p.c_q <= 8) return launch_fwd<D, 8, TO, WIDE>(p, part, q, k, v, w, o, m, l, s);
    return launch_fwd<D, 11, TO, WIDE>(p, part, q, k, v, w, o, m, l, s);
}

template <int CQT> size_t split_bytes(const Problem &p) {
    constexpr int BQ = NW * wave_rows(CQT);
    const int share = fwd_share<BQ>(p);
    return share ? (size_t)p.B * p.H * fwd_wgs<BQ>(p, share) * BQ * (p.d + 4) * sizeof(float) : 0;
}

template <bool WIDE>
hipError_t pick_shape(const Problem &p, int out_dt, const void *q, const void *k, const void *v,
                      const float *w, void *o, float *m, float *l, hipStream_t s, float *part) {
    if (p.d == 128) {
        if (out_dt == CONVATTN_BF16) return pick_cq<128, bf16_t, WIDE>(p, part, q, k, v, w, o, m, l, s);
        return pick_cq<128, float, WIDE>(p, part, q, k, v, w, o, m, l, s);
    }
    if (p.d == 32) {
        if (out_dt == CONVATTN_BF16) return pick_cq<32, bf16_t, WIDE>(p, part, q, k, v, w, o, m, l, s);
        return pick_cq<32, float, WIDE>(p, part, q, k, v, w, o, m, l, s);
    }
    if (out_dt == CONVATTN_BF16) return pick_cq<64, bf16_t, WIDE>(p, part, q, k, v, w, o, m, l, s);
    return pick_cq<64, float, WIDE>(p, part, q, k, v, w, o, m, l, s);
}

}  // namespace

// This file is compiled twice, the second time (CONVATTN_FWD_WIDE) for the windows of 17 key taps, so that the two sets of instances
// build in parallel.
#ifdef CONVATTN_FWD_WIDE
hipError_t mfma_fwd_wide(const Problem &p, int out_dt, const void *q, const void *k, const void *v,
                         const float *w, void *o, float *m, float *l, hipStream_t s, float *part) {
    return pick_shape<true>(p, out_dt, q, k, v, w, o, m, l, s, part);
}
#else
size_t mfma_fwd_split_bytes(const Problem &p) {
    return p.c_q <= 3   ? split_bytes<3>(p)
           : p.c_q <= 6 ? split_bytes<6>(p)
           : p.c_q <= 7 ? split_bytes<7>(p)
           : p.c_q <= 8 ? split_bytes<8>(p)
                        : split_bytes<11>(p);
}

hipError_t mfma_fwd(const Problem &p, int out_dt, const void *q, const void *k, const void *v,
                    const float *w, void *o, float *m, float *l, hipStream_t s, float *part) {
    if (p.c_k > kSparseMaxCk) return mfma_fwd_wide(p, out_dt, q, k, v, w, o, m, l, s, part);
    return pick_shape<false>(p, out_dt, q, k, v, w, o, m, l, s, part);
}
#endif

}  // namespace convattn
