// Whole backward of conv-attention on bf16 MFMA (gfx950), windows of 7 to 11 query taps at head dimension 128 (instances of 7, 8
// and 11 tap slots): the score chain stays in registers.  (Other windows run the three-role kernel of bwd_chain3_mfma.hip,
// which shares this file's building blocks through chain_common.hpp; the per-(batch, head) dC scale
// kernels of both live here.)
//
// Key-stationary: a workgroup of 8 waves owns 128 keys of one (batch, head) and walks down the
// query rows in tiles of 32.  Pair p (waves p and p+4, one SIMD) owns keys c0 = k0 + 32p .. c0+31
// for dK and dS, c0-8 .. c0+23 for dV and dW.  Everything between the two products of a tile is
// kept in the layout "lane = query row, registers = 4 keys" that the accumulators of
// S^T = K Q^T come out in (lane n of fragment f holds row r0 + 2n + f):
//   producer (waves 0-3): dP^T = V dO^T - D; S^T (raw, pre-masked, packed to fp16); the
//       convolution as Toeplitz MFMAs whose B operand is the packed S^T itself, row-shifted by
//       DPP moves (rows above the tile come from the previous tile's registers);
//       P = exp2(C - LSE), dC = P dP.  P (bf16), dC and S (fp16) go to LDS as [row][key] tiles.
//   consumer (waves 4-7), one tile behind: dV^T += dO^T P and dW += dC^T S with the operands read
//       back through LDS transpose reads; two tiles behind: dS^T by flipped-band MFMAs over the
//       packed dC^T (rows below a tile come from the next tile, hence the extra tile of delay),
//       dS -> workspace (bf16 blocks of 32 rows x 32 keys in the order the lanes hold them) and
//       -> LDS, dK^T += Q^T dS.
// One workgroup barrier per tile; Q and dO tiles go from global memory straight into LDS (buffer
// loads with the LDS modifier, one tile ahead), in a layout that serves both the 128-bit row
// fragment reads of the producers and the 64-bit transpose reads of dV / dK (see ChainLds).
// The transposed convolution of a pair's 32 keys needs dC on the 16 keys after them as well: every
// pair computes that block itself.
//
// dW[a][b] = sum_i sum_j dC[i][j] S_m[i+a-pq][j+b-pk] is computed as G_a = dC^T S(rows shifted by
// a), a [key j] x [key j'] product contracted over the rows on the matrix cores; only its
// diagonals |j'-j| <= pk are wanted, so a 16-key block of j needs two 16-key blocks of j' and both
// blocks of j add into the same two accumulators per tap.  The diagonals are summed once, after
// the last tile.
//
// dC is carried as fp16 times a power of two chosen per (batch, head) from the magnitudes of dO
// and V (dc_scale), which makes the backward linear in dO over the whole range of bf16: dK, dV, dW
// and (in the dQ product) dQ are multiplied by its inverse when they are stored.
#include <type_traits>

#include "chain_common.hpp"

namespace convattn {
namespace {

using namespace chain;


constexpr int NT = 2 * NP * 64;  // 512 threads
#if !defined(CONVATTN_CHAIN_UNIT) || CONVATTN_CHAIN_UNIT == 3
#define CONVATTN_CHAIN_UNIT_IS_ALL 1
#else
#define CONVATTN_CHAIN_UNIT_IS_ALL 0
#endif
constexpr int kPF = 3;   // dO^T / Q^T fragments read ahead of their MFMAs in the dV / dK phases

// One role of the workgroup (ROLE 0 = producer waves, 1 = consumer waves).  The two roles have
// disjoint register sets of 256 each and are both inlined into the kernel: as called functions
// each wave would save and restore the 112 callee-saved vector registers it uses through scratch
// memory (0.47 GB written and read back per C3 launch, 7 % of the kernel's time).
// WANT: bit 0 = dK and dV, bit 1 = dS (for dQ) and dW; the passes behind the separate dK / dV and dQ + dW
// operations leave the other half out.
template <int D, int CQT, typename TO, int ROLE, int WANT>
__device__ __forceinline__ void chain_role(const CHAIN_CONST_AS ChainArgs *args_in) {
    // the pointer arrives in vector registers; it is the same in every lane, and as a scalar the
    // arguments are fetched with scalar loads into scalar registers
    const unsigned long long av = reinterpret_cast<unsigned long long>(args_in);
    const unsigned long long as =
        ((unsigned long long)(unsigned int)__builtin_amdgcn_readfirstlane((int)(av >> 32)) << 32) |
        (unsigned int)__builtin_amdgcn_readfirstlane((int)(unsigned int)av);
    const ChainArgs args = *reinterpret_cast<const CHAIN_CONST_AS ChainArgs *>(as);
    const Problem p = args.p;
    const bf16_t *__restrict__ Q = args.Q, *__restrict__ K = args.K, *__restrict__ V = args.V, *__restrict__ dO = args.dO;
    const float *__restrict__ Dl = args.Dl, *__restrict__ LSE = args.LSE, *__restrict__ W = args.W;
    const float *__restrict__ dc_scale = args.dc_scale;
    TO *__restrict__ dK = static_cast<TO *>(args.dK), *__restrict__ dV = static_cast<TO *>(args.dV);
    bf16_t *__restrict__ dS_ws = args.dS_ws;
    float *__restrict__ dW_part = args.dW_part;
    const int n_rt = args.n_rt;
    static_assert(D == 128 && CQT > 6, "the three-role kernel serves the others");
    using Lds = ChainLds<D, CQT>;
    constexpr int KS = D / 32, DB = D / 16;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, n = lane & 15;
    constexpr bool producer = ROLE == 0;
    constexpr bool WANT_KV = (WANT & 1) != 0, WANT_QW = (WANT & 2) != 0;
    const int pr = wave & (NP - 1);

    auto q_slot = [&](int t) { return smem + Lds::q_off + (t & 3) * Lds::tile_bytes; };
    auto g_slot = [&](int t) { return smem + Lds::g_off + (t % 3) * Lds::tile_bytes; };
    auto stat_slot = [&](int t) { return reinterpret_cast<float *>(smem + Lds::stat_off + (t & 1) * (2 * BR * 4)); };
    unsigned char *pair_base = smem + Lds::pair_off + pr * Lds::pair_bytes;
    unsigned char *s_ring = pair_base;
    auto c_stage = [&](int t) { return pair_base + Lds::s_bytes + (t & 1) * (BR * CST); };
    auto p_stage = [&](int t) { return pair_base + Lds::s_bytes + Lds::c_bytes + (t & 1) * (BR * PST); };
    unsigned char *ds_tile = pair_base + Lds::s_bytes + Lds::c_bytes + Lds::p_bytes;

    // x = head, y = batch, z = key tile: the first key tiles see the most rows and go first
    const int h = blockIdx.x, b = blockIdx.y;
    // (SPLIT: instances of their own, the others are up to 2 % slower with the parts' bounds at run time)
    constexpr bool SPLIT = (WANT & 4) != 0;
    const ChainSpan span = SPLIT ? chain_span(p, blockIdx.z, args.share) : ChainSpan{(int)blockIdx.z, 0, 0, 0, 1};
    const int k0 = span.kb * BKW, c0 = k0 + pr * WK;
    const int pk = p.pk, cq = p.c_q, ck = p.c_k;
    const bool causal = p.causal != 0;
    const size_t bh = (size_t)b * p.H + h;
    const bf16_t *Qb = Q + bh * p.Nq * D;
    const bf16_t *dOb = dO + bh * p.Nq * D;
    const float *lse_b = LSE + bh * p.Nq;
    const float *dl_b = Dl + bh * p.Nq;
    // dC scale (a power of two): given by the caller, or, without one, taken from D = rowsum(dO O) of
    // this (batch, head): D is linear in dO and of the magnitude of dP, so s |D|max ~ 2^8 keeps dC in
    // the normal range of fp16 whatever the magnitude of dO is
    float dcs, dcs_log2;
    if (dc_scale) {
        dcs = dc_scale[2 * bh];
        dcs_log2 = dc_scale[2 * bh + 1];
    } else {
        dcs_log2 = dc_scale_log2_from_d(dl_b, p.Nq, tid, NT, reinterpret_cast<float *>(smem + Lds::stat_off));
        dcs = exp2f(dcs_log2);
    }

    // Causal: rows before the first key this workgroup touches (k0 - 8) see none of its keys.
    const int t_begin = SPLIT ? span.len * span.part / span.parts : 0, t_end = SPLIT ? span.len * (span.part + 1) / span.parts : 0;
    const int r_begin = SPLIT ? (span.first_rt + t_begin) * BR : causal ? (max(0, k0 - 8) / BR) * BR : 0;
    const int n_tiles = SPLIT ? t_end - t_begin : (p.Nq - r_begin + BR - 1) / BR;
    // The window of the last tile's rows reaches into the tile after it, whose dC is computed here too where it is
    // another workgroup's: n_scored tiles have scores and dC, n_tiles of them everything else.
    const int n_scored = n_tiles + (SPLIT && t_end < span.len ? 1 : 0);
    // this workgroup's partial dK / dV, or null: it writes the results itself
    float *kv_part = SPLIT && span.parts > 1 ? args.kv_part + (bh * gridDim.z + blockIdx.z) * (2 * BKW * D) : nullptr;
    // masks are needed next to the diagonal, at both ends of the key axis and past the last row
    const bool always_edge = c0 < 8 || c0 + 40 > p.Nk;
    auto is_edge = [&](int r0) { return always_edge || (causal && r0 < c0 + 64) || r0 + BR > p.Nq; };
    // no (row, key) pair of the tile is visible: only its scores are needed, by the tile below
    auto is_skipped = [&](int r0) { return causal && r0 + BR - 1 < c0 - 8; };

    // Q / dO tiles: global memory -> LDS without passing through registers.  A tile is 2 KBT units
    // of 1 KB (KBT of Q, then KBT of dO; unit 2 ks + f = the 16 row pairs of one k-step and parity);
    // wave w issues the units w, w + 8, ...  Lane l of a load fills chunk position l % 4 of row pair
    // l / 4.  Rows after the last query row are outside the descriptor's range and arrive as zeros.
    // (Inline assembly: for the builtin the compiler makes every later LDS read wait for the load,
    // as it cannot tell the tile slots apart; the wait is written out before the barrier instead.)
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    constexpr int KBT = Lds::tile_bytes / 1024;
    static_assert(KBT == 2 * KS, "one unit per k-step and row parity");
    auto dma_rsrc = [&](const bf16_t *ptr) {
        const unsigned long long a = reinterpret_cast<unsigned long long>(ptr);
        return (i32x4){(int)(unsigned int)a, (int)(unsigned int)(a >> 32), p.Nq * D * 2, 0x00020000};
    };
    const i32x4 q_dma = dma_rsrc(Qb), g_dma = dma_rsrc(dOb);
    const unsigned int lds0 = (unsigned int)(unsigned long long)(__attribute__((address_space(3))) unsigned char *)smem;
    auto fetch_tile = [&](int t) {
        const int ln = (int)opaque((unsigned int)lane);
#pragma unroll
        for (int j0 = 0; j0 < 2 * KBT; j0 += 2 * NP) {
            const int j = j0 + wave, m = j / KBT, kb = j - m * KBT;
            const int row = 2 * (ln >> 2) + (kb & 1), chunk = (kb >> 1) * 4 + ((ln & 3) ^ ((ln >> 4) & 3));
            const int voff = ((r_begin + t * BR + row) * D + chunk * 8) * 2;
            const unsigned int dst = lds0 + (m ? Lds::g_off + (t % 3) * Lds::tile_bytes : Lds::q_off + (t & 3) * Lds::tile_bytes) + kb * 1024;
            const i32x4 rsrc = m ? g_dma : q_dma;
            // (M0 is written here and read by the load that follows; nothing else of this kernel uses it,
            // and it is not declared clobbered: the compiler keeps no value in M0 across an asm statement)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                         :: "s"(dst), "v"(voff), "s"(rsrc) : "memory");
        }
    };
    // Every tile this wave has asked for is in LDS (to be followed by the workgroup barrier).  Vector
    // memory operations complete in the order of their issue: `younger` = the global stores the wave
    // has issued since the tile loads (the dS block of an iteration: NDB * 2), which need not be waited for.
    // The count holds only while a wave issues exactly those stores, and no other vector memory operation,
    // between its loads and this wait: the statistics loads are issued before the tile loads.
    auto tiles_landed = [&](bool younger) {
        if (younger) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NDB * 2) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    static_assert((2 * KBT) % (2 * NP) == 0, "whole units per wave");
    // LSE and D of a tile: loaded by the first 32 lanes of the first producer wave one iteration before they
    // are written to LDS.
    constexpr bool STAT_ROLE = ROLE == 0;
    // (a wave-uniform test, i.e. a branch: the other waves of the role must not even touch `ls` / `dd`, whose
    // reuse as load destinations makes the compiler wait for every outstanding vector memory operation of the
    // wave, the dS stores of the last iteration among them)
    const bool stat_wave = STAT_ROLE && wave == 0;
    float ls = 0.f, dd = 0.f;
    auto load_stats = [&](int r0) {
        if constexpr (STAT_ROLE) {
            if (stat_wave) {
                // raw values: arithmetic on them here would wait for the loads in this iteration
                const int tt = (int)opaque((unsigned int)lane);
                ls = 1e30f; dd = 0.f;  // rows past the end: exp2(C - LSE) = 0
                if (tt < BR && r0 + tt < p.Nq) { ls = lse_b[r0 + tt]; dd = dl_b[r0 + tt]; }
            }
        }
    };
    auto stage_stats = [&](int t) {
        if constexpr (STAT_ROLE) {
            if (stat_wave) {
                const int tt = (int)opaque((unsigned int)lane);
                float *st = stat_slot(t);
                if (tt < BR) { st[tt] = ls * kLog2e - dcs_log2; st[BR + tt] = dd; }
            }
        }
    };
    // Lane parts of the fragment addresses inside a tile.  Row fragment (producers): row 2n + f,
    // chunk 4 ks + g: + f KB + 2 ks KB.  Transposed fragment (consumers): rows 4g + n/4 (+ 16 hi),
    // 8 bytes at byte column 32 db + 8 (n % 4): see read_tr_t for the constant part.
    auto row_frag_off = [&] { return (unsigned int)(n * 64 + ((g ^ ((n >> 2) & 3)) << 4)); };
    auto tr_frag_off = [&] {
        return (unsigned int)(((n >> 2) & 1) * 1024 + (2 * g + (n >> 3)) * 64 + ((((n >> 1) & 1) ^ (g >> 1)) << 4) + (n & 1) * 8);
    };
    auto read_tr_t = [&](const unsigned char *lane_ptr, int db) {   // (db: a constant after unrolling)
        // rows + 16: row pair + 8, whose chunk positions are those of this one with bit 1 flipped
        bf16x4 lo = lds_tr64(lane_ptr + (db >> 1) * 2048 + ((db & 1) << 5));
        bf16x4 hi = lds_tr64(lane_ptr + (db >> 1) * 2048 + (((db & 1) ^ 1) << 5) + 512);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };

    // Set-up: every global load of it is issued before the first wait (the first tile, K / V
    // fragments, the rows above the first tile, the window's weights), so that it costs one round
    // trip to memory instead of several.
    fetch_tile(0);
    load_stats(r_begin);
    // bands of the window (direct: times scale * log2 e, the convolved scores come out in log2 units; flipped:
    // times the softmax scale); the first barrier of the tile loop publishes them
    if constexpr (Lds::compact_bands)
        band_tab_build<CQT>(smem + Lds::band_off, W + (size_t)h * cq * ck, cq, ck, pk, p.scale * kLog2e, p.scale, tid, NT);
    // lane's part of a band's address: the tap slot is a constant offset from one address register
    const unsigned int band_lane = Lds::compact_bands ? band_tab_lane_off(g, n) : lane * 16;
    auto read_band = [&](const unsigned char *lane_ptr, int slot) {   // (slot: a constant after unrolling)
        if constexpr (Lds::compact_bands) return band_tab_read(lane_ptr + slot * Lds::band_slot);
        else return *reinterpret_cast<const f16x8 *>(lane_ptr + slot * Lds::band_slot);
    };

    if constexpr (producer) {
        // ================================ producer ================================
        const bf16_t *Kb = K + bh * p.Nk * D;
        const bf16_t *Vb = V + bh * p.Nk * D;
        const unsigned char *bands = smem + opaque((unsigned int)Lds::band_off + band_lane);
        bf16x8 kf[NSB][KS];  // K rows c0-16 .. c0+47
        bf16x8 vf[NCB][KS];  // V rows c0-8 .. c0+39
#pragma unroll
        for (int kb = 0; kb < NSB; ++kb)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                kf[kb][ks] = __builtin_bit_cast(bf16x8, load_row16_nb<D>(Kb, c0 - 16 + kb * 16 + n, p.Nk, ks * 32 + g * 8));
#pragma unroll
        for (int kb = 0; kb < NCB; ++kb)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                vf[kb][ks] = __builtin_bit_cast(bf16x8, load_row16_nb<D>(Vb, c0 - 8 + kb * 16 + n, p.Nk, ks * 32 + g * 8));

        // Q rows of the 32 rows above the first tile
        bf16x8 q_above[2][KS];
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                q_above[f][ks] = __builtin_bit_cast(bf16x8, load_row16_nb<D>(Qb, r_begin - BR + 2 * n + f, p.Nq, ks * 32 + g * 8));
        // (ready-made fragments: one KB per tap slot, the slots dealt out to the four waves)
        if constexpr (!Lds::compact_bands)
            for (int t = pr; t < CQT; t += NP)
                *reinterpret_cast<f16x8 *>(smem + Lds::band_off + t * 1024 + lane * 16) =
                    band_frag<CQT>(t, W + (size_t)h * cq * ck, cq, ck, pk, g, n, false, p.scale * kLog2e);
        stage_stats(0);
        load_stats(r_begin + BR);

        // Every pair computes the C / dP / dC block after its own keys (keys c0+24 .. c0+39) itself, and with it
        // the fourth S^T block.
        {
        constexpr int PNSB = NSB, PNCB = NCB;
        // packed fp16 scores of the previous tile: [block][fragment][dword]
        unsigned int prev_pd[NSB][2][2];

        // S^T of the 32 rows r0 .. r0+31 (ring tile tp), pre-masked, packed and stored for dW
        auto s_phase = [&](int r0, int tp, unsigned int (&pd)[NSB][2][2], auto edge_tag, auto &&load_qf) {
            constexpr bool EDGE = decltype(edge_tag)::value;
            f32x4 acc[NSB][2];
#pragma unroll
            for (int kb = 0; kb < PNSB; ++kb)
#pragma unroll
                for (int f = 0; f < 2; ++f) acc[kb][f] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                bf16x8 qf[2];
#pragma unroll
                for (int f = 0; f < 2; ++f) qf[f] = load_qf(f, ks);
#pragma unroll
                for (int kb = 0; kb < PNSB; ++kb)
#pragma unroll
                    for (int f = 0; f < 2; ++f) acc[kb][f] = mfma_bf16(kf[kb][ks], qf[f], acc[kb][f]);
            }
            const int rbase = (tp * BR) % Lds::ring_rows;
#pragma unroll
            for (int kb = 0; kb < PNSB; ++kb)
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    if constexpr (EDGE) {
                        if (causal) {
                            const int qpos = r0 + 2 * n + f, key0 = c0 - 16 + kb * 16 + 4 * g;
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (key0 + r > qpos) acc[kb][f][r] = 0.f;
                        }
                    }
                    // rounded exactly as the forward rounds its scores: P = exp2(C - LSE)
                    // only sums to one over a row if C is the C the forward's LSE was taken from
                    const u32x2 two = pack_scores_f16(acc[kb][f]);
                    pd[kb][f][0] = two[0];
                    pd[kb][f][1] = two[1];
                    if (WANT_QW && kb < 3) {
                        const int rr = rbase + 2 * n + f;
                        *reinterpret_cast<u32x2 *>(s_ring + (rr >= Lds::ring_rows ? rr - Lds::ring_rows : rr) * SST + (kb * 16 + 4 * g) * 2) =
                            (u32x2){pd[kb][f][0], pd[kb][f][1]};
                    }
                }
        };

        // the 32 rows above the first tile: their scores are the window's halo for tile 0
        {
            s_phase(r_begin - BR, 0, prev_pd, std::true_type{}, [&](int f, int ks) { return q_above[f][ks]; });
        }
        for (int it = 0; it <= n_tiles + 1; ++it) {
            const int r0 = r_begin + it * BR;
            tiles_landed(false);
            __syncthreads();
            // (the LSE / D loads before the tile loads: the wait above is for the youngest loads of the wave)
            if (it + 1 < n_scored) stage_stats(it + 1);
            load_stats(r0 + 2 * BR);
            if (it + 1 < n_scored) fetch_tile(it + 1);
            // dC of a tile that has none (entirely above the diagonal, or the one after the last):
            // zeros, so that the consumers read every tile alike
            auto zero_dc = [&] {
                // (address from the lane index afresh: nothing of this rare path stays in a register)
                const unsigned int ln = opaque((unsigned int)lane);
                unsigned char *Cs = c_stage(it) + 2 * (ln & 15) * CST + (ln >> 4) * 8;
#pragma unroll
                for (int cb = 0; cb < PNCB; ++cb)
#pragma unroll
                    for (int ob = 0; ob < 2; ++ob)
                        *reinterpret_cast<u32x2 *>(Cs + ob * CST + cb * 32) = (u32x2){0u, 0u};
            };
            if (it == n_scored) zero_dc();
            if (it >= n_scored) continue;

            auto ptile = [&](auto edge_tag, auto full_tag) {
                constexpr bool EDGE = decltype(edge_tag)::value;
                constexpr bool FULL = decltype(full_tag)::value;
                // row fragments: lane n of fragment f reads row 2n + f, 16 bytes at column 32 ks + 8 g
                const unsigned char *Qs = smem + opaque((unsigned int)(q_slot(it) - smem) + row_frag_off());
                const unsigned char *Gs = smem + opaque((unsigned int)(g_slot(it) - smem) + row_frag_off());
                __builtin_amdgcn_s_setprio(1);
                f32x4 dp[NCB][2];
                float2 l2 = {0.f, 0.f};
                if constexpr (FULL) l2 = *reinterpret_cast<const float2 *>(stat_slot(it) + 2 * n);
                // ---- S^T ----
                unsigned int pd[NSB][2][2];
                s_phase(r0, it + 1, pd, edge_tag, [&](int f, int ks) {
                    return *reinterpret_cast<const bf16x8 *>(Qs + f * 1024 + ks * 2048);
                });
                                if constexpr (FULL) {
                    unsigned char *Cs = c_stage(it), *Ps = p_stage(it);
                    // ---- convolution: C^T block cb from score blocks cb (k slots 0..3 of a lane
                    // group) and cb+1 (4..7).  Operand of row offset delta = DL - (CQT-1): fragment
                    // f = delta & 1 shifted s = (f - delta) / 2 lanes down; it serves output parity
                    // 0 with tap slot DL and parity 1 with tap slot DL - 1. ----
                    f32x4 c[NCB][2];
#pragma unroll
                    for (int cb = 0; cb < PNCB; ++cb) {
                        c[cb][0] = (f32x4){-l2.x, -l2.x, -l2.x, -l2.x};
                        c[cb][1] = (f32x4){-l2.y, -l2.y, -l2.y, -l2.y};
                    }
                    f16x8 tf_prev = (f16x8)(_Float16)0.f;
                    static_for<CQT + 1>([&](auto DL) {
                        constexpr int t0 = decltype(DL)::value;
                        constexpr int delta = t0 - (CQT - 1);
                        constexpr int f = delta & 1, s = (f - delta) / 2;
                        f16x8 tf_cur = tf_prev;
                        if constexpr (t0 < CQT) tf_cur = read_band(bands, t0);
                        unsigned int sh[NSB][2];
#pragma unroll
                        for (int kb = 0; kb < PNSB; ++kb)
#pragma unroll
                            for (int dw = 0; dw < 2; ++dw) sh[kb][dw] = win_up<s>(prev_pd[kb][f][dw], pd[kb][f][dw]);
#pragma unroll
                        for (int cb = 0; cb < PNCB; ++cb) {
                            const u32x4 bv = {sh[cb][0], sh[cb][1], sh[cb + 1][0], sh[cb + 1][1]};
                            if constexpr (t0 < CQT) c[cb][0] = mfma_f16(tf_cur, __builtin_bit_cast(f16x8, bv), c[cb][0]);
                            if constexpr (t0 >= 1) c[cb][1] = mfma_f16(tf_prev, __builtin_bit_cast(f16x8, bv), c[cb][1]);
                        }
                        tf_prev = tf_cur;
                    });
#pragma unroll
                    for (int kb = 0; kb < PNSB; ++kb)
#pragma unroll
                        for (int f = 0; f < 2; ++f) { prev_pd[kb][f][0] = pd[kb][f][0]; prev_pd[kb][f][1] = pd[kb][f][1]; }
                    // ---- dP^T = V dO^T - D, after the convolution: the shifted score windows are no
                    // longer live then (with dP first, some instances of the kernel needed scratch) ----
                    {
                        const float2 d2 = *reinterpret_cast<const float2 *>(stat_slot(it) + BR + 2 * n);
#pragma unroll
                        for (int cb = 0; cb < PNCB; ++cb) {
                            dp[cb][0] = (f32x4){-d2.x, -d2.x, -d2.x, -d2.x};
                            dp[cb][1] = (f32x4){-d2.y, -d2.y, -d2.y, -d2.y};
                        }
#pragma unroll
                        for (int ks = 0; ks < KS; ++ks) {
                            bf16x8 gf[2];
#pragma unroll
                            for (int f = 0; f < 2; ++f)
                                gf[f] = *reinterpret_cast<const bf16x8 *>(Gs + f * 1024 + ks * 2048);
#pragma unroll
                            for (int cb = 0; cb < PNCB; ++cb)
#pragma unroll
                                for (int f = 0; f < 2; ++f) dp[cb][f] = mfma_bf16(vf[cb][ks], gf[f], dp[cb][f]);
                        }
                    }
                                        // ---- P = exp2(C - LSE) (times the dC scale), dC = P dP ----
                    static_for<PNCB>([&](auto CB) {
                        constexpr int cb = decltype(CB)::value;
                        __builtin_amdgcn_s_setprio(0);
#pragma unroll
                        for (int ob = 0; ob < 2; ++ob) {
                            f32x4 prob, dc;
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                prob[r] = fast_exp2(c[cb][ob][r]);
                                dc[r] = prob[r] * dp[cb][ob][r];
                            }
                            if constexpr (EDGE) {
                                const int qpos = r0 + 2 * n + ob;
#pragma unroll
                                for (int r = 0; r < 4; ++r) {
                                    const int key = c0 - 8 + cb * 16 + 4 * g + r;
                                    if (key < 0 || key >= p.Nk || (causal && key > qpos)) { prob[r] = 0.f; dc[r] = 0.f; }
                                }
                            }
                            *reinterpret_cast<u32x2 *>(Cs + (2 * n + ob) * CST + (cb * 16 + 4 * g) * 2) =
                                (u32x2){pack_f16_rtz(dc[0], dc[1]), pack_f16_rtz(dc[2], dc[3])};
                            if constexpr (WANT_KV && cb < 2) {
                                bf16x4 pv;
#pragma unroll
                                for (int r = 0; r < 4; ++r) pv[r] = (bf16_t)prob[r];
                                *reinterpret_cast<bf16x4 *>(Ps + (2 * n + ob) * PST + (cb * 16 + 4 * g) * 2) = pv;
                            }
                        }
                    });
                } else {
#pragma unroll
                    for (int kb = 0; kb < PNSB; ++kb)
#pragma unroll
                        for (int f = 0; f < 2; ++f) { prev_pd[kb][f][0] = pd[kb][f][0]; prev_pd[kb][f][1] = pd[kb][f][1]; }
                    zero_dc();
                }
            };
            if (is_skipped(r0)) ptile(std::true_type{}, std::false_type{});
            else if (is_edge(r0)) ptile(std::true_type{}, std::true_type{});
            else ptile(std::false_type{}, std::true_type{});
        }
        }
        __syncthreads();  // the consumers' barrier before they hand over their dW accumulators
        __syncthreads();  // ... and the one after it
        // ---- dW partial of this workgroup: G[m][n] of half x belongs to key tap b = n - m + 16 x - 8 + pk;
        // the sum runs over the pair groups, the halves and the diagonals' elements in a fixed order.
        // S was raw, so * scale; dC was scaled, so / dcs. ----
        static_assert(2 * CQT * 2 * 1024 <= NP * ChainLds<D, CQT>::pair_bytes, "room for the dW accumulators");
        // Four lanes per tap (pair group, half), each adds its diagonal's elements in index order; the
        // four sums are added as (0 + 1) + (2 + 3).
        const int ntap = cq * ck;
        for (int q = tid; WANT_QW && (q >> 2) < ntap; q += NT / 2) {
            const int tap = q >> 2, a = tap / ck, bb = tap - a * ck, t = a + CQT - cq;
            const int pgi = (q >> 1) & 1, x = q & 1;
            const float *red = reinterpret_cast<const float *>(smem + Lds::pair_off) + ((pgi * CQT + t) * 2 + x) * 256;
            float sum = 0.f;
#pragma unroll
            for (int m = 0; m < 16; ++m) {
                const int nn = bb + m - 16 * x + 8 - pk;
                const float val = red[m * 16 + min(max(nn, 0), 15)];
                if (nn >= 0 && nn < 16) sum += val;
            }
            sum += __shfl_xor(sum, 1);
            sum += __shfl_xor(sum, 2);
            if ((q & 3) == 0) dW_part[(bh * gridDim.z + blockIdx.z) * ntap + tap] = sum * p.scale / dcs;
        }
    } else {
        // ================================ consumer ================================
        const float *w_head = W + (size_t)h * cq * ck;
        // flipped bands, after the direct ones
        unsigned char *bands = smem + opaque((unsigned int)Lds::band_off + CQT * Lds::band_slot + band_lane);
        if constexpr (!Lds::compact_bands)
            for (int t = pr; t < CQT; t += NP)
                *reinterpret_cast<f16x8 *>(bands + t * 1024) = band_frag<CQT>(t, w_head, cq, ck, pk, g, n, true, p.scale);
        stage_stats(0);
        load_stats(r_begin + BR);
        // dW: a unit is the key blocks of two pairs (pair group) times one tap slot; every wave takes one pair
        // group and half of the tap slots, in one pass (two for more than 8 tap slots: the operands of a
        // pass are in registers three key blocks deep).
        // (an odd number of slots: the second wave of a group multiplies its last one twice and drops the copy)
        constexpr int NPASS = CQT > 8 ? 2 : 1, TH = (CQT + 1) / 2, NU = TH / NPASS;   // units per pass
        static_assert(NU * NPASS == TH, "whole units per pass");
        int dw_pg[NPASS], dw_t[NPASS];   // pair group and first tap slot
#pragma unroll
        for (int ps = 0; ps < NPASS; ++ps) { dw_pg[ps] = pr >> 1; dw_t[ps] = (pr & 1) * TH + ps * NU; }
        f32x4 acc_k[NDB][DB], acc_v[2][DB];
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                acc_k[m][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
                acc_v[m][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
        f32x4 acc_w[TH][2];
#pragma unroll
        for (int t = 0; t < TH; ++t) acc_w[t][0] = acc_w[t][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
        unsigned int prev_dc[NCB][2][2];
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
            for (int f = 0; f < 2; ++f) prev_dc[cb][f][0] = prev_dc[cb][f][1] = 0u;
        const int n_kt = (SPLIT ? (p.Nk + 8 + BKW - 1) / BKW : (int)gridDim.z) * NP, kt = span.kb * NP + pr;
        // (causal: the pair's first block is row tile kt - 1)
        bf16_t *ds_pair = dS_ws + (bh * (size_t)chain_ds_block_off(causal, n_rt, n_kt) + (size_t)chain_ds_block_off(causal, n_rt, kt) -
                                   chain_ds_first_rt(causal, kt)) * (WK * BR);
        bool ds_stored = false;  // the last iteration stored a dS block (after its tile loads)
        for (int it = 0; it <= n_tiles + 1; ++it) {
            tiles_landed(ds_stored);
            ds_stored = false;
            __syncthreads();
            // (the LSE / D loads before the tile loads: the counted wait above relies on that order)
            if (it + 1 < n_scored) stage_stats(it + 1);
            load_stats(r_begin + (it + 2) * BR);
            if (it + 1 < n_scored) fetch_tile(it + 1);
            const int u = it - 1, v = it - 2;
            const int r0u = r_begin + u * BR, r0v = r_begin + v * BR;
            const bool u_in = it >= 1 && u < n_tiles;
            const bool u_ok = u_in && !is_skipped(r0u);
            const bool v_ok = it >= 2 && !is_skipped(r0v);

            // Order of the iteration: dV (operands of the staged tiles only, so the first MFMAs
            // start while the dC loads are in flight), dS, dW (independent of dS: its MFMAs cover
            // the round trip of dS through LDS), dK.
            if (WANT_KV && u_ok) {
                const unsigned char *Ps = smem + opaque((unsigned int)(p_stage(u) - smem) + tr_lane_off(PST, g, n));
                const unsigned char *Gs = smem + opaque((unsigned int)(g_slot(u) - smem) + tr_frag_off());
                __builtin_amdgcn_s_setprio(1);
                // ---- dV^T += dO^T P (keys c0-8 .. c0+23) ----
                // the dO^T fragment of head-dim block db + PF is read while block db is multiplied: the
                // MFMAs of PF blocks cover the LDS latency
                constexpr int PF = kPF;
                bf16x8 pf[2], gq[PF + 1];
#pragma unroll
                for (int cb = 0; cb < 2; ++cb) pf[cb] = read_tr(Ps, PST, cb * 16);
#pragma unroll
                for (int db = 0; db < PF && db < DB; ++db) gq[db] = read_tr_t(Gs, db);
                static_for<DB>([&](auto DBI) {
                    constexpr int db = decltype(DBI)::value;
                    if constexpr (db + PF < DB) {
                        gq[(db + PF) % (PF + 1)] = read_tr_t(Gs, db + PF);
                        SCHED_DS_READ_ID(2, 60 + db);
                    }
#pragma unroll
                    for (int cb = 0; cb < 2; ++cb) acc_v[cb][db] = mfma_bf16(gq[db % (PF + 1)], pf[cb], acc_v[cb][db]);
                    SCHED_MFMA_ID(2, 60 + db);
                });
            }
            // packed dC^T of tile u, as the producer's lanes held it (zeros when the tile has none)
            unsigned int cur_dc[NCB][2][2];
            {
                // read unconditionally: the producer writes zeros for a tile without dC; what the first
                // iteration reads (nothing written yet) is dropped before any use
                const unsigned char *Cl = smem + opaque((unsigned int)(c_stage(max(u, 0)) - smem) + 2 * n * CST + 4 * g * 2);
                // the block after the pair's own keys: the third block of the pair's own stage
                const unsigned char *Cn = Cl + 2 * 32;
#pragma unroll
                for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
                    for (int f = 0; f < 2; ++f) {
                        const u32x2 t2 = *reinterpret_cast<const u32x2 *>(cb < 2 ? Cl + f * CST + cb * 32 : Cn + f * CST);
                        cur_dc[cb][f][0] = t2[0];
                        cur_dc[cb][f][1] = t2[1];
                    }
            }
            if (v_ok) {
                const bool edge = is_edge(r0v);
                bf16_t *ds_blk = ds_pair + (size_t)(r0v / BR) * (WK * BR);
                __builtin_amdgcn_s_setprio(2);
                // ---- dS^T of tile v: rows below it come from tile v+1.  Operand of row offset
                // e = parity + (CQT-1 - tap slot): fragment e & 1 shifted e >> 1 lanes up. ----
                f32x4 ds[NDB][2];
#pragma unroll
                for (int sb = 0; sb < NDB; ++sb) ds[sb][0] = ds[sb][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
                // flipped bands: the fragment of step e + 2 is read during step e (two steps of MFMAs
                // cover the LDS latency; read one step ahead, every step waited for its band)
                auto band_of = [&](int e) { return read_band(bands, CQT - 1 - e); };
                f16x8 tbq[4];   // bands of steps e-1 .. e+2
                tbq[0] = band_of(0);
                tbq[1] = band_of(CQT >= 2 ? 1 : 0);
                tbq[2] = tbq[3] = tbq[0];
                static_for<CQT + 1>([&](auto E) {
                    constexpr int e = decltype(E)::value, f = e & 1, s = e >> 1;
                    // tap slot CQT-1-e for parity 0 (this step's band), CQT-e for parity 1 (the last step's)
                    if constexpr (e + 2 <= CQT - 1) tbq[(e + 2) % 4] = band_of(e + 2);
                    const f16x8 tb_cur = tbq[e % 4], tb_prev = tbq[(e + 3) % 4];
                    unsigned int sh[NCB][2];
#pragma unroll
                    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
                        for (int dw = 0; dw < 2; ++dw) sh[cb][dw] = win_down<s>(prev_dc[cb][f][dw], cur_dc[cb][f][dw]);
#pragma unroll
                    for (int sb = 0; sb < NDB; ++sb) {
                        const u32x4 bv = {sh[sb][0], sh[sb][1], sh[sb + 1][0], sh[sb + 1][1]};
                        if constexpr (e <= CQT - 1) ds[sb][0] = mfma_f16(tb_cur, __builtin_bit_cast(f16x8, bv), ds[sb][0]);
                        if constexpr (e >= 1) ds[sb][1] = mfma_f16(tb_prev, __builtin_bit_cast(f16x8, bv), ds[sb][1]);
                    }
                });
#pragma unroll
                for (int sb = 0; sb < NDB; ++sb)
#pragma unroll
                    for (int ob = 0; ob < 2; ++ob) {
                        if (edge && causal) {
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (c0 + sb * 16 + 4 * g + r > r0v + 2 * n + ob) ds[sb][ob][r] = 0.f;
                        }
                        bf16x4 sv;
#pragma unroll
                        for (int r = 0; r < 4; ++r) sv[r] = (bf16_t)ds[sb][ob][r];
                        // block layout [row parity][key half][16 row pairs][16 keys]: the 64 lanes of a store
                        // write 512 contiguous bytes
                        if constexpr (WANT_QW) {
                            // (non-temporal: read once, by another kernel; kept out of the L2)
                            __builtin_nontemporal_store(__builtin_bit_cast(u32x2, sv),
                                                        reinterpret_cast<u32x2 *>(ds_blk + ((ob * 2 + sb) * 16 + n) * 16 + 4 * g));
                            ds_stored = true;
                        }
                        if constexpr (WANT_KV) *reinterpret_cast<bf16x4 *>(ds_tile + (2 * n + ob) * PST + (sb * 16 + 4 * g) * 2) = sv;
                    }
            }
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
                for (int f = 0; f < 2; ++f) { prev_dc[cb][f][0] = cur_dc[cb][f][0]; prev_dc[cb][f][1] = cur_dc[cb][f][1]; }
            // ---- dW, key blocks jb = 0..3 of the pairs 2 pg and 2 pg + 1 (block jb = dC block jb & 1 of
            // pair 2 pg + jb / 2, keys k0 + 64 pg - 8 + 16 jb ..), tap slots t_lo .. t_lo + TH - 1:
            // G_t[j][j'] += sum_rows dC[row][j] S[row + t - (CQT-1)][j'] with j' in the score block
            // 8 keys before the dC block (x = 0) and the one 8 keys after it (x = 1) ----
            if (WANT_QW && u_in) static_for<NPASS>([&](auto PS) {
                constexpr int ps = decltype(PS)::value;
                const int pg = dw_pg[ps], t_lo = dw_t[ps];
                // Ring rows of this lane's two transpose reads at the wave's first tap slot: tile row 0
                // at tap slot 0 is ring row wbase; the TH tap slots are consecutive rows (mod the ring's rows).
                const int wbase = ((u + 1) * BR - (CQT - 1) + Lds::ring_rows) % Lds::ring_rows;
                const unsigned int c_lane = opaque(tr_lane_off(CST, g, n));
                const unsigned int ring0 = Lds::pair_off + 2 * pg * Lds::pair_bytes + 4 * (n & 3) * 2;
                unsigned int a_lo[NU], a_hi[NU];
#pragma unroll
                for (int tt = 0; tt < NU; ++tt) {
                    const unsigned int ra = wbase + 4 * g + (n >> 2) + min(t_lo + tt, CQT - 1), rb = ra + 16;
                    a_lo[tt] = opaque(ring0 + min(ra, ra - Lds::ring_rows) * SST);
                    a_hi[tt] = opaque(ring0 + min(rb, rb - Lds::ring_rows) * SST);
                }
                // score block jb' = 0..4 of the group: block jb' & 1 (or 2 for the last) of pair 2 pg + jb' / 2
                // (blocks 0..3: a constant offset from the lane's address; block 4 is block 0 of the pair
                // after the group or, for the last group, block 2 of its second pair: a[][] of it apart)
                const unsigned int off4 = pg == NP / 2 - 1 ? Lds::pair_bytes + 64 : 2 * Lds::pair_bytes;
                unsigned int a4_lo[NU], a4_hi[NU];
#pragma unroll
                for (int tt = 0; tt < NU; ++tt) { a4_lo[tt] = a_lo[tt] + off4; a4_hi[tt] = a_hi[tt] + off4; }
                auto s_frag = [&](auto JBP, int tt) {
                    constexpr int jbp = decltype(JBP)::value;
                    constexpr int off = (jbp >> 1) * Lds::pair_bytes + (jbp & 1) * 32;
                    bf16x4 l4, h4;
                    if constexpr (jbp < 4) {
                        l4 = lds_tr64(smem + a_lo[tt] + off);
                        h4 = lds_tr64(smem + a_hi[tt] + off);
                    } else {
                        l4 = lds_tr64(smem + a4_lo[tt]);
                        h4 = lds_tr64(smem + a4_hi[tt]);
                    }
                    return __builtin_bit_cast(f16x8, __builtin_shufflevector(l4, h4, 0, 1, 2, 3, 4, 5, 6, 7));
                };
                // dC^T block jb of the group (a pair whose tile is entirely above the diagonal holds zeros)
                auto c_frag = [&](int jb) {
                    const int dq = jb >> 1;
                    return __builtin_bit_cast(
                        f16x8, read_tr(smem + Lds::pair_off + 2 * pg * Lds::pair_bytes + Lds::s_bytes + (u & 1) * (BR * CST) +
                                           c_lane + dq * Lds::pair_bytes, CST, (jb & 1) * 16));
                };
                // Software pipeline over the four key blocks: the operands of block jb + 1 are read
                // while block jb is multiplied.  Every tap slot of the wave is multiplied, also the
                // zero taps in front of a narrow window (their sums are not used).
                f16x8 af = c_frag(0), b0[NU], b1[NU];
#pragma unroll
                for (int tt = 0; tt < NU; ++tt) {
                    b0[tt] = s_frag(std::integral_constant<int, 0>{}, tt);
                    b1[tt] = s_frag(std::integral_constant<int, 1>{}, tt);
                }
                static_for<4>([&](auto JB) {
                    constexpr int jb = decltype(JB)::value;
                    f16x8 af_n = af, b2[NU];
#pragma unroll
                    for (int tt = 0; tt < NU; ++tt) b2[tt] = b1[tt];
                    if constexpr (jb < 3) {
                        af_n = c_frag(jb + 1);
#pragma unroll
                        for (int tt = 0; tt < NU; ++tt) b2[tt] = s_frag(std::integral_constant<int, jb + 2>{}, tt);
                        SCHED_DS_READ_ID(2 + 2 * NU, 40 + 4 * ps + jb);
                    }
#pragma unroll
                    for (int tt = 0; tt < NU; ++tt) {
                        acc_w[ps * NU + tt][0] = mfma_f16(af, b0[tt], acc_w[ps * NU + tt][0]);
                        acc_w[ps * NU + tt][1] = mfma_f16(af, b1[tt], acc_w[ps * NU + tt][1]);
                    }
                    SCHED_MFMA_ID(2 * NU, 40 + 4 * ps + jb);
                    af = af_n;
#pragma unroll
                    for (int tt = 0; tt < NU; ++tt) { b0[tt] = b1[tt]; b1[tt] = b2[tt]; }
                });
            });
            if (WANT_KV && v_ok) {
                const unsigned char *Qs = smem + opaque((unsigned int)(q_slot(v) - smem) + tr_frag_off());
                const unsigned char *Dsl = smem + opaque((unsigned int)(ds_tile - smem) + tr_lane_off(PST, g, n));
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_s_setprio(1);
                // ---- dK^T += Q^T dS ----
                {
                    constexpr int PF = kPF;
                    bf16x8 sf[2], qq[PF + 1];
                    // (Q^T does not depend on the dS tile: its first fragments are on their way first)
#pragma unroll
                    for (int db = 0; db < PF && db < DB; ++db) qq[db] = read_tr_t(Qs, db);
#pragma unroll
                    for (int sb = 0; sb < 2; ++sb) sf[sb] = read_tr(Dsl, PST, sb * 16);
                    static_for<DB>([&](auto DBI) {
                        constexpr int db = decltype(DBI)::value;
                        if constexpr (db + PF < DB) {
                            qq[(db + PF) % (PF + 1)] = read_tr_t(Qs, db + PF);
                            SCHED_DS_READ_ID(2, 70 + db);
                        }
#pragma unroll
                        for (int sb = 0; sb < 2; ++sb) acc_k[sb][db] = mfma_bf16(qq[db % (PF + 1)], sf[sb], acc_k[sb][db]);
                        SCHED_MFMA_ID(2, 70 + db);
                    });
                }
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
            }
            __builtin_amdgcn_s_setprio(0);
        }
        // ---- dW accumulators of this wave to LDS as [pair group][tap slot][x][m][n], once every
        // wave is done with the tiles ----
        __syncthreads();
        float *red = reinterpret_cast<float *>(smem + Lds::pair_off);
#pragma unroll
        for (int ps = 0; ps < NPASS; ++ps)
#pragma unroll
            for (int tt = 0; tt < NU; ++tt)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (WANT_QW && dw_t[ps] + tt < CQT)
                            red[(((dw_pg[ps] * CQT + dw_t[ps] + tt) * 2 + x) * 16 + 4 * g + r) * 16 + n] = acc_w[ps * NU + tt][x][r];
        __syncthreads();  // the producers add the dW partial up while the consumers store dK and dV

        // ---- stores: lane = key, 4 consecutive head-dim columns per block ----
        const float inv = 1.f / dcs;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int key_k = c0 + m * 16 + n;
            const int key_v = c0 - 8 + m * 16 + n;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const int col = db * 16 + 4 * g;
                if (SPLIT && WANT_KV && kv_part) {
                    float *dst = kv_part + (pr * WK + m * 16 + n) * D + col;
                    *reinterpret_cast<f32x4 *>(dst) = acc_k[m][db] * inv;
                    *reinterpret_cast<f32x4 *>(dst + BKW * D) = acc_v[m][db] * inv;
                    continue;
                }
                if (WANT_KV && key_k < p.Nk) {
                    TO *dst = dK + (bh * p.Nk + key_k) * D + col;
                    if constexpr (sizeof(TO) == 2) {
                        bf16x4 ov;
#pragma unroll
                        for (int r = 0; r < 4; ++r) ov[r] = (bf16_t)(acc_k[m][db][r] * inv);
                        *reinterpret_cast<bf16x4 *>(dst) = ov;
                    } else {
                        *reinterpret_cast<f32x4 *>(dst) = acc_k[m][db] * inv;
                    }
                }
                if (WANT_KV && key_v >= 0 && key_v < p.Nk) {
                    TO *dst = dV + (bh * p.Nk + key_v) * D + col;
                    if constexpr (sizeof(TO) == 2) {
                        bf16x4 ov;
#pragma unroll
                        for (int r = 0; r < 4; ++r) ov[r] = (bf16_t)(acc_v[m][db][r] * inv);
                        *reinterpret_cast<bf16x4 *>(dst) = ov;
                    } else {
                        *reinterpret_cast<f32x4 *>(dst) = acc_v[m][db] * inv;
                    }
                }
            }
        }

    }  // consumer
}

template <int D, int CQT, typename TO, int WANT>
__global__ __launch_bounds__(NT) void bwd_chain_kernel(ChainArgs args) {
    // `args` is the whole argument segment; the roles read it from there
#if defined(__HIP_DEVICE_COMPILE__)
    const CHAIN_CONST_AS ChainArgs *ap =
        (const CHAIN_CONST_AS ChainArgs *)__builtin_amdgcn_kernarg_segment_ptr();
#else
    const ChainArgs *ap = &args;
#endif
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < NP) chain_role<D, CQT, TO, 0, WANT>(ap);
    else chain_role<D, CQT, TO, 1, WANT>(ap);
}

#if CONVATTN_CHAIN_UNIT_IS_ALL
// amax|dO| and amax|V| of one (batch, head) -> {s, log2 s}, s the power of two that brings
// sqrt(d) * amax|dO| * amax|V| (a few times a typical |dP|) to about 2^12.  Two steps: kScaleChunks
// workgroups per (batch, head) leave their maxima in `part`, one thread per (batch, head) finishes.
__global__ __launch_bounds__(256) void dc_scale_partial_kernel(int Nq, int Nk, int d, const bf16_t *__restrict__ dO,
                                                               const bf16_t *__restrict__ V, float *__restrict__ part) {
    const size_t bh = (size_t)blockIdx.z * gridDim.y + blockIdx.y;   // y = head, z = batch
    __shared__ float red[2][4];
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        const size_t cnt = (size_t)(which ? Nk : Nq) * d / 8;   // 16-byte pieces of the slab
        const size_t per = (cnt + kScaleChunks - 1) / kScaleChunks;
        const size_t lo = blockIdx.x * per, hi = lo + per < cnt ? lo + per : cnt;
        const u32x4 *src = reinterpret_cast<const u32x4 *>((which ? V : dO) + bh * (which ? Nk : Nq) * (size_t)d);
        unsigned int m = 0;
        for (size_t i = lo + threadIdx.x; i < hi; i += 256) {
            const u32x4 v = src[i];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                m = max(m, (v[j] << 16) & 0x7fffffffu);
                m = max(m, v[j] & 0x7fff0000u);
            }
        }
        // NaN / Inf inputs (exponent all ones) are left out of the maximum: they poison the results anyway
        const float mx = wave_max(m < 0x7f800000u ? __uint_as_float(m) : 0.f);
        if ((threadIdx.x & 63) == 0) red[which][threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x < 2)
        part[(bh * kScaleChunks + blockIdx.x) * 2 + threadIdx.x] =
            fmaxf(fmaxf(red[threadIdx.x][0], red[threadIdx.x][1]), fmaxf(red[threadIdx.x][2], red[threadIdx.x][3]));
}
__global__ void dc_scale_finish_kernel(int n_bh, int d, const float *__restrict__ part, float *__restrict__ out) {
    const int bh = blockIdx.x * blockDim.x + threadIdx.x;
    if (bh >= n_bh) return;
    float a = 0.f, v = 0.f;
    for (int c = 0; c < kScaleChunks; ++c) {
        a = fmaxf(a, part[((size_t)bh * kScaleChunks + c) * 2]);
        v = fmaxf(v, part[((size_t)bh * kScaleChunks + c) * 2 + 1]);
    }
    write_dc_scale(d, a, v, out + 2 * bh);
}

#endif

template <int D, int CQT, typename TO, int WANT>
hipError_t launch_chain(const Problem &p, const void *q, const void *k, const void *v, const void *d_o,
                        const float *Dl, const float *lse, const float *w, const float *dc_scale, void *dk,
                        void *dv, void *ds_ws, float *dw_part, int share, float *kv_part, hipStream_t s) {
    auto kern = bwd_chain_kernel<D, CQT, TO, WANT>;
    constexpr int lds = ChainLds<D, CQT>::total;
    static_assert(lds <= 160 * 1024, "LDS budget");
    hipError_t e = set_max_lds_once<bwd_chain_kernel<D, CQT, TO, WANT>>(lds);
    if (e != hipSuccess) return e;
    dim3 grid(p.H, p.B, chain_wgs(p, share));
    ChainArgs args{p, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, (const bf16_t *)d_o, Dl, lse, w,
                   dc_scale, dk, dv, (bf16_t *)ds_ws, dw_part, chain_row_tiles(p), share, kv_part};
    kern<<<grid, NT, lds, s>>>(args);
    return hipGetLastError();
}

template <int D, typename TO, int WANT>
hipError_t pick_cq(const Problem &p, const void *q, const void *k, const void *v, const void *d_o,
                   const float *Dl, const float *lse, const float *w, const float *dc_scale, void *dk, void *dv,
                   void *ds_ws, float *dw_part, int share, float *kv_part, hipStream_t s) {
    // (the others run the three-role kernel of bwd_chain3_mfma.hip; forward + backward of B4 H16 N2048 d128 7x7 in 8 slots 682 us,
    // in 7 665)
#define CALL(CQT) launch_chain<D, CQT, TO, WANT>(p, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s)
    return p.c_q <= 7 ? CALL(7) : p.c_q == 8 ? CALL(8) : CALL(11);
#undef CALL
}

template <int WANT>
hipError_t pick_out(const Problem &p, int out_dt, const void *q, const void *k, const void *v, const void *d_o,
                      const float *Dl, const float *lse, const float *w, const float *dc_scale, void *dk, void *dv,
                      void *ds_ws, float *dw_part, int share, float *kv_part, hipStream_t s) {
    if (out_dt == CONVATTN_BF16) return pick_cq<128, bf16_t, WANT>(p, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s);
    return pick_cq<128, float, WANT>(p, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s);
}

}  // namespace


#if CONVATTN_CHAIN_UNIT_IS_ALL
hipError_t mfma_dc_scale(const Problem &p, const void *d_o, const void *v, float *dc_scale, hipStream_t s) {
    // dc_scale holds {s, log2 s} per (batch, head), then the partial maxima
    float *part = dc_scale + (size_t)p.B * p.H * 2;
    dc_scale_partial_kernel<<<dim3(kScaleChunks, p.H, p.B), 256, 0, s>>>(p.Nq, p.Nk, p.d, (const bf16_t *)d_o,
                                                                          (const bf16_t *)v, part);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? dc_scale_finish(p, dc_scale, s) : e;
}
hipError_t dc_scale_finish(const Problem &p, float *dc_scale, hipStream_t s) {
    dc_scale_finish_kernel<<<dim3((p.B * p.H + 255) / 256), 256, 0, s>>>(p.B * p.H, p.d, dc_scale + (size_t)p.B * p.H * 2, dc_scale);
    return hipGetLastError();
}
#endif

// This file is compiled once per value of CONVATTN_CHAIN_UNIT (1 = dK and dV only, 2 = dS and dW
// only, 3 = everything, 7 = everything with split row ranges), so that the three sets of instances build in parallel.
#ifndef CONVATTN_CHAIN_UNIT
#define CONVATTN_CHAIN_UNIT 3
#endif
#if CONVATTN_CHAIN_UNIT == 1
#define CHAIN_ENTRY mfma_bwd_chain_kv
#elif CONVATTN_CHAIN_UNIT == 7
#define CHAIN_ENTRY mfma_bwd_chain_split
#elif CONVATTN_CHAIN_UNIT == 2
#define CHAIN_ENTRY mfma_bwd_chain_qw
#else
#define CHAIN_ENTRY mfma_bwd_chain_all
#endif
hipError_t CHAIN_ENTRY(const Problem &p, int out_dt, const void *q, const void *k, const void *v,
                       const void *d_o, const float *Dl, const float *lse, const float *w,
                       const float *dc_scale, void *dk, void *dv, void *ds_ws, float *dw_part, int share, float *kv_part, hipStream_t s) {
    return pick_out<CONVATTN_CHAIN_UNIT>(p, out_dt, q, k, v, d_o, Dl, lse, w, dc_scale, dk, dv, ds_ws, dw_part, share, kv_part, s);
}

}  // namespace convattn
