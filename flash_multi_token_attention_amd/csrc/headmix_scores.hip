// One-pass backward of head-mixing attention (gfx950): dQ, dK, dV and the gradient of the mixing matrix.
//
//   S_h' = Q_h' K_h'^T,  Z_h = scale sum_h' w[h][h'] S_h',  P_h = exp(Z_h - LSE_h),  dP_h = dO_h V_h^T,
//   dZ_h = P_h (dP_h - D_h),  dS_h' = scale sum_h w[h][h'] dZ_h,  dw[h][h'] = scale sum dZ_h S_h',
//   dQ_h' = dS_h' K_h',  dK_h' = dS_h'^T Q_h',  dV_h = P_h^T dO_h.
//
// The head mix couples all heads of a (row, key) pair, the last three products couple all keys (or
// rows) of a head.  Kept in one workgroup, their accumulators (2 H d floats per key) leave room for 16
// keys only, and every byte of Q and dO is then loaded for 16 keys at a time.  So the pass is cut between
// the two: headmix_scores_kernel computes P and dS once per (row, key) pair and writes them as bf16
// blocks of 32 rows x 32 keys (the operand precision of the products that follow); dQ = dS K is
// the product kernel of the window backward (bwd_dq_rows.hip, same block layout) and
// headmix_dkdv_kernel takes dV = P^T dO and dK = dS^T Q from one walk over the blocks of 128 keys.
#include "dq_rows.hpp"
#include "headmix_common.hpp"
#include "reduce_common.hpp"

namespace convattn {
namespace {

using namespace headmix;
constexpr int SC_BLK = kBlock;

// 8 waves of 256 registers.  16 heads: 32 rows x 16 keys per step, two tile buffers; 32 heads: 16 rows x 32 keys, one.
template <int H, int D> struct ScoreTile : Tile<H, 8, H == 16 ? 32 : 16> {
    using B = Tile<H, 8, H == 16 ? 32 : 16>;
    static constexpr int SPW = 2 * B::HPW;                  // heads of a wave in the score phase
    static constexpr int ROOM = B::R * (D * 2 + 16);        // a head's rows while they are turned
    // LDS per head: scores, then dP (then dZ in its place) at a distance that fits the instructions' offsets; +4 floats as in Tile
    static constexpr int DP = B::R * B::KT, HS = 2 * DP + 4, NBUF = H == 16 ? 2 : 1;
    static constexpr bool STATS_LDS = D >= 64;               // LSE and D of the tile rows: registers are short
    static constexpr int w_off = NBUF * H * HS, wt_off = w_off + H * B::WST, st_off = wt_off + H * B::WST,
                         sp_off = st_off + (STATS_LDS ? 2 * B::R * B::WST : 0),   // H = 32: the split of w and its transpose
                         used = sp_off * 4 + (H == 32 ? 2 * kSplitBytes : 0), lds = used > B::WAVES * ROOM ? used : B::WAVES * ROOM;
    // chunks (one head, 16 keys) of K or V rows in registers, and how many of them stay in flight during the mixing phase
    static constexpr int RING = H == 16 || D < 128 ? 4 : 2, AHEAD = D == 128 ? (H == 16 ? 2 : 0) : 4;
    // (B4 H16 N4096 d128: 2 / 3 / 4 chunks in flight 1.27 / 1.33 / 1.32 ms; without the two orders of scores and mix 1.34)
    // Key steps ahead of its use that a step's K and V are asked for, a dword of each 128-byte line, so that the fragment loads
    // find them in the L2: the workgroups of an XCD walk the same keys in step, so all of them wait for each of its misses
    // (a fragment load comes two chunks ahead, and the memory takes a whole step under the stores of the blocks).  The
    // workgroups of an XCD take the heads in turn; a value is dropped two steps later, when it has arrived.
    // B4 H16 N4096 d128, us: none 1231, 3 steps 1100, 6 steps 1095.
    static constexpr int ASK = 6;
    static_assert(SPW * B::KB % RING == 0, "a chunk's registers are the same in every step");
};

struct ScoreArgs {
    int B, N, causal, n_rt32, n_kt;
    Plan plan;
    float scale;
    const bf16_t *Q, *KF, *VF, *dO;   // KF, VF: fragment order
    const float *W, *lse, *Dl;
    bf16_t *P, *dS;      // blocks; the same address where P is not wanted: a lane writes an element of P, then of dS, in this order
    float *dw_part;      // [n_wg][H][H], or null
};

// AHEAD: K and V are asked for ahead of their use, and short tiles walked down (score_ahead)
template <int H, int D, bool AHEAD>
__global__ __launch_bounds__((ScoreTile<H, D>::WAVES * 64)) void headmix_scores_kernel(ScoreArgs a) {
    using T = ScoreTile<H, D>;
    constexpr int RB = T::RB, R = T::R, KT = T::KT, KB = T::KB, NQ = T::NQ, RW = T::RW, HS = T::HS, DP = T::DP, SPW = T::SPW,
                  HB = T::HB, KS = D / 32, NCH = SPW * KB;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    float *lds = reinterpret_cast<float *>(smem);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane_id = threadIdx.x & 63;
    const int id = share_of_workgroup(a.plan), N = a.N;
    if (id < 0) return;
    // score phase: the first half of the waves takes S = Q K^T, the second half dP = dO V^T, SPW heads each
    const int mat = wave / (T::WAVES / 2), h0 = (wave - mat * (T::WAVES / 2)) * SPW;

    // w of the mix and its transpose, with the scales of the two products, in LDS (read as four k steps at a time:
    // k slot g of step s is head 4g + s)
    for (int i = threadIdx.x; i < H * H; i += T::WAVES * 64) {
        const float w = a.W[i];
        lds[T::w_off + (i / H) * T::WST + i % H] = w * (a.scale * kLog2e);
        lds[T::wt_off + (i % H) * T::WST + i / H] = w * a.scale;
        if constexpr (H == 32) {
            put_split(lds + T::sp_off, i / H, i % H, w * (a.scale * kLog2e));
            put_split(smem + T::sp_off * 4 + kSplitBytes, i % H, i / H, w * a.scale);
        }
    }
    f32x4 acc_w[HB][HB];
#pragma unroll
    for (int x = 0; x < HB; ++x)
#pragma unroll
        for (int y = 0; y < HB; ++y) acc_w[x][y] = (f32x4){0.f, 0.f, 0.f, 0.f};

    for (int x_pos = id * a.plan.share, x_end = (int)min((long long)x_pos + a.plan.share, (long long)a.B * a.plan.entry_len); x_pos < x_end;) {
    const Segment sg = find_segment(a.plan, id, x_pos, AHEAD);
    const int b = sg.b, rt = sg.rt, n_steps = sg.len();
    x_pos += n_steps;
    int lane = lane_id;
    asm volatile("" : "+v"(lane));   // (no registers for what could be kept from segment to segment)
    const int tid = wave * 64 + lane, g = lane >> 4, n = lane & 15, i0 = rt * R;
    const size_t bo = (size_t)b * H * N * D;

    // ---- resident: Q or dO fragments of this wave's heads ----
    bf16x8 qf[SPW][RB][KS];
#pragma unroll
    for (int t = 0; t < SPW; ++t)
        turn_rows<T, D>(qf[t], (mat ? a.dO : a.Q) + bo + (size_t)(h0 + t) * N * D, i0, N, smem + wave * T::ROOM);
    lds_barrier();   // the score tiles go where the other waves' rows are
    // ---- the mixing phase: lane (g, n) = heads 4g .. 4g+3 of each block of 16, tile row lr, keys 4q .. 4q+3 ----
    const int lr = wave * RW + (n & (RW - 1)), q4 = n / RW;
    const int row = T::row(i0, lr);
    // (rows past the last: P = exp2(-1e30) = 0, so nothing of them is in dS, dV, dK or dw)
    float *st_l = lds + T::st_off;
    f32x4 lse_r[HB], dl_r[HB];
    if constexpr (T::STATS_LDS) {
        for (int i = tid; i < R * H; i += T::WAVES * 64) {
            const int hh = i / R, lr2 = i % R, rr = T::row(i0, lr2);
            const size_t o = ((size_t)b * H + hh) * N + min(rr, N - 1);
            st_l[lr2 * T::WST + hh] = rr < N ? a.lse[o] * -kLog2e : -1e30f;
            st_l[(R + lr2) * T::WST + hh] = a.Dl[o];
        }
    } else {
#pragma unroll
        for (int hb = 0; hb < HB; ++hb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const size_t o = ((size_t)b * H + 16 * hb + 4 * g + r) * N + min(row, N - 1);
                lse_r[hb][r] = row < N ? a.lse[o] * -kLog2e : -1e30f;
                dl_r[hb][r] = a.Dl[o];
            }
    }
    const float *wf_l = lds + T::w_off + n * T::WST + 4 * g, *wb_l = lds + T::wt_off + n * T::WST + 4 * g;
    // ---- score phase, in chunks of one head and 16 keys whose rows are loaded two chunks ahead ----
    bf16x8 kf[T::RING][KS];
    const int n_t16 = a.n_rt32 * 2;
    const bf16_t *frag = (mat ? a.VF : a.KF) + ((size_t)b * H + h0) * n_t16 * KS * 512;
    auto load_chunk = [&](int step, int c) {
        const bf16_t *kp = frag + ((size_t)(c / KB) * n_t16 + step * KB + c % KB) * KS * 512;   // (the same in all lanes)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kf[c % T::RING][ks] = *at<bf16x8>(kp, (unsigned)lane * 16 + ks * 1024);
    };
    auto score_chunk = [&](float *S, int c) {
        const int t = c / KB, kb = c % KB;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) s = mfma_bf16(kf[c % T::RING][ks], qf[t][rb][ks], s);
            *reinterpret_cast<f32x4 *>(S + mat * DP + (h0 + t) * HS + (rb * 16 + n) * KT + 4 * T::slot(rb * 16 + n, 4 * kb + g)) = s;
        }
    };

    // ---- mixing phase of one step ----
    const int pos = lr * KT + 4 * T::slot(lr, q4);
    // element of a block for this lane: [row parity][key half][row pair][16 keys]
    const int brow = row & 31;
    const unsigned out = 2 * ((((brow & 1) * 2 + (q4 >> 2)) * 16 + (brow >> 1)) * 16 + 4 * (q4 & 3) + 4 * g * SC_BLK);
    const int key_max = a.causal ? min(row, N - 1) : N - 1;   // last key the row sees
    auto mix = [&](float *S, int step) {
        float *dP = S + DP;
        const int j0 = step * KT;
        f32x4 z[HB][4];   // starting at -LSE
        auto start = [&] {
#pragma unroll
            for (int x = 0; x < HB; ++x) {
                f32x4 nlse = lse_r[x];
                if constexpr (T::STATS_LDS) nlse = *reinterpret_cast<const f32x4 *>(st_l + lr * T::WST + 16 * x + 4 * g);
#pragma unroll
                for (int t = 0; t < 4; ++t) z[x][t] = nlse;
            }
        };
        auto mix_fp32 = [&] {
#pragma unroll
            for (int y = 0; y < HB; ++y) {
                f32x4 wf[HB];
#pragma unroll
                for (int x = 0; x < HB; ++x) wf[x] = *reinterpret_cast<const f32x4 *>(wf_l + 16 * x * T::WST + 16 * y);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(S + (16 * y + 4 * g + s) * HS + pos);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int x = 0; x < HB; ++x) z[x][t] = mfma4(wf[x][s], v[t], z[x][t]);
                }
            }
        };
        start();
        if constexpr (H == 32) {
            mix_split<T>(z, S, pos, g, lds + T::sp_off, lane);
            if (has_nan(z)) {
                start();
                mix_fp32();
            }
        } else {
            mix_fp32();
        }
        // masks only where a key of the tile is past the tile's first row or past the last key
        if ((a.causal && j0 + KT - 1 > i0) || j0 + KT > N) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bool dead = j0 + 4 * q4 + t > key_max;
#pragma unroll
                for (int x = 0; x < HB; ++x)
#pragma unroll
                    for (int r = 0; r < 4; ++r) z[x][t][r] = dead ? kNegInf : z[x][t][r];
            }
        }
        const int kt = j0 / 32;
        const long long blk = chain_ds_block_off(a.causal != 0, a.n_rt32, kt) + i0 / 32 - chain_ds_first_rt(a.causal != 0, kt);
        // blocks of all heads side by side: [batch][block][head][1024]
        const long long n_blk = chain_ds_block_off(a.causal != 0, a.n_rt32, a.n_kt);
        const size_t first = ((size_t)b * n_blk + blk) * H * SC_BLK;
        const int half = KT == 16 ? (step & 1) * 256 : 0;    // steps of 16 keys: the second half of the block's keys
        bf16_t *p_out = a.P + first + half, *ds_out = a.dS + first + half;
#pragma unroll
        for (int x = 0; x < HB; ++x) {
            f32x4 dl = dl_r[x];
            if constexpr (T::STATS_LDS) dl = *reinterpret_cast<const f32x4 *>(st_l + (R + lr) * T::WST + 16 * x + 4 * g);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float *dz = dP + (16 * x + 4 * g + r) * HS + pos;
                f32x4 d = *reinterpret_cast<const f32x4 *>(dz);
                bf16x4 pb;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float p = fast_exp2(z[x][t][r]);
                    pb[t] = (bf16_t)p;
                    d[t] = p * (d[t] - dl[r]);
                    z[x][t][r] = d[t];
                }
                *reinterpret_cast<f32x4 *>(dz) = d;
                __builtin_nontemporal_store(__builtin_bit_cast(u32x2, pb), at<u32x2>(p_out, out + (16 * x + r) * SC_BLK * 2));
            }
        }
        f32x4 ds[HB][4];
        auto dmix_fp32 = [&] {
#pragma unroll
            for (int x = 0; x < HB; ++x) {
#pragma unroll
                for (int t = 0; t < 4; ++t) ds[x][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int y = 0; y < HB; ++y) {
                    const f32x4 wb = *reinterpret_cast<const f32x4 *>(wb_l + 16 * x * T::WST + 16 * y);
#pragma unroll
                    for (int s = 0; s < 4; ++s)
#pragma unroll
                        for (int t = 0; t < 4; ++t) ds[x][t] = mfma4(wb[s], z[y][t][s], ds[x][t]);
                }
            }
        };
        if constexpr (H == 32) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {   // (a key at a time: two took up to 16 registers that are not there)
                const f32x4 z0 = z[0][t], z1 = z[HB - 1][t];
                const Split sp[1] = {split8({z0[0], z0[1], z0[2], z0[3], z1[0], z1[1], z1[2], z1[3]})};
                ds[0][t] = ds[HB - 1][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
                mfma_split<1>({&ds[0][t], &ds[HB - 1][t]}, smem + T::sp_off * 4 + kSplitBytes, lane, sp);
            }
            if (has_nan(ds)) {
                asm volatile("" ::: "memory");   // (dZ from where it was put: kept in registers it would be in everyone's way)
#pragma unroll
                for (int x = 0; x < HB; ++x)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const f32x4 dz = *reinterpret_cast<const f32x4 *>(dP + (16 * x + 4 * g + r) * HS + pos);
#pragma unroll
                        for (int t = 0; t < 4; ++t) z[x][t][r] = dz[t];
                    }
                dmix_fp32();
            }
        } else {
            dmix_fp32();
        }
#pragma unroll
        for (int x = 0; x < HB; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                bf16x4 db;
#pragma unroll
                for (int t = 0; t < 4; ++t) db[t] = (bf16_t)ds[x][t][r];
                __builtin_nontemporal_store(__builtin_bit_cast(u32x2, db), at<u32x2>(ds_out, out + (16 * x + r) * SC_BLK * 2));
            }
        // dw += dZ S^T over the wave's own 64 pairs: lane n = head of either operand
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < RW * NQ / 4; ++i) {
            // (quads in the order in which they lie: the sum runs over all of them)
            const int o = n * HS + wave * RW * KT + i * 16 + 4 * g;
            f32x4 za[HB], sb[HB];
#pragma unroll
            for (int x = 0; x < HB; ++x) {
                za[x] = *reinterpret_cast<const f32x4 *>(dP + 16 * x * HS + o);
                sb[x] = *reinterpret_cast<const f32x4 *>(S + 16 * x * HS + o);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int x = 0; x < HB; ++x)
#pragma unroll
                    for (int y = 0; y < HB; ++y) acc_w[x][y] = mfma4(za[x][e], sb[y][e], acc_w[x][y]);
        }
    };

    // the chunks of `step` into S; the first AHEAD ones of step `next` are loaded on the way
    auto scores = [&](float *S, int step, int next) {
#pragma unroll
        for (int c = T::AHEAD; c < T::RING; ++c) load_chunk(step, c);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            score_chunk(S, c);
            if (c + T::RING < NCH) load_chunk(step, c + T::RING);
            else if (c + T::RING - NCH < T::AHEAD) load_chunk(next, c + T::RING - NCH);
        }
    };
#pragma unroll
    for (int c = 0; c < T::AHEAD; ++c) load_chunk(sg.step(0), c);
    const auto later = [&](int i) { return sg.step(min(i, n_steps - 1)); };
    if constexpr (T::NBUF == 2) {
        // One barrier per step.  Of the two waves of a SIMD one takes the scores of the next step first, the other the mix of
        // this one, so that one's LDS and vector work runs under the other's products.
        scores(lds, sg.step(0), later(1));
        lds_barrier();
        unsigned asked[2] = {0, 0};
        for (int u = 0; u < n_steps; ++u) {
            if constexpr (AHEAD) {
                if (wave == 0) {
                    static_assert(H == 16 && KB * KS * 8 == 32, "a line of a head's K or V per lane");
                    const size_t tile = ((size_t)b * H + (blockIdx.x >> 3) % H) * n_t16 + later(u + T::ASK);
                    asm volatile("" ::"v"(asked[0]));
                    asked[0] = asked[1];
                    asked[1] = *reinterpret_cast<const unsigned *>((lane < 32 ? a.KF : a.VF) + tile * KS * 512 + lane % 32 * 64);
                }
            }
            float *cur = lds + (u & 1) * H * HS, *nxt = lds + ((u + 1) & 1) * H * HS;
            const bool first = wave < T::WAVES / 2, more = u + 1 < n_steps;
            const int next = later(u + 1), ahead = later(u + 2);
            if (more && first) scores(nxt, next, ahead);
            mix(cur, sg.step(u));
            if (more && !first) scores(nxt, next, ahead);
            lds_barrier();
        }
    } else {
        for (int u = 0; u < n_steps; ++u) {
            scores(lds, sg.step(u), later(u + 1));
            lds_barrier();
            mix(lds, sg.step(u));
            lds_barrier();
        }
    }
    }   // segments

    // ---- the workgroup's dw partial: the waves' accumulators added in wave order ----
    if (a.dw_part) {
        const int g = lane_id >> 4, n = lane_id & 15;
#pragma unroll
        for (int x = 0; x < HB; ++x)
#pragma unroll
            for (int y = 0; y < HB; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r) lds[(wave * H + 16 * x + 4 * g + r) * H + 16 * y + n] = acc_w[x][y][r];
        lds_barrier();
        float *part = a.dw_part + (size_t)id * H * H;
        for (int i = threadIdx.x; i < H * H; i += T::WAVES * 64) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < T::WAVES; ++w) s += lds[w * H * H + i];
            part[i] = s * a.scale;
        }
    }
}

// dw[h][h'] = sum of the partials in a fixed order: a workgroup takes 16 entries, 16 threads per entry each
// add every 16th partial, the sixteen sums are added in order.
__device__ __forceinline__ void dw_sum(int n_part, int hh, const float *__restrict__ part, float *__restrict__ dW, int block,
                                       float (*red)[17]) {
    const int e = threadIdx.x & 15, c = threadIdx.x >> 4, idx = block * 16 + e;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    int q = c;
    for (; q + 48 < n_part; q += 64) {
        s0 += part[(size_t)q * hh + idx];
        s1 += part[(size_t)(q + 16) * hh + idx];
        s2 += part[(size_t)(q + 32) * hh + idx];
        s3 += part[(size_t)(q + 48) * hh + idx];
    }
    for (; q < n_part; q += 16) s0 += part[(size_t)q * hh + idx];
    red[c][e] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    if (threadIdx.x < 16) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) s += red[i][threadIdx.x];
        dW[block * 16 + threadIdx.x] = s;
    }
}
__global__ __launch_bounds__(256) void headmix_dw_sum_kernel(int n_part, int hh, const float *__restrict__ part,
                                                             float *__restrict__ dW) {
    __shared__ float red[16][17];
    dw_sum(n_part, hh, part, dW, blockIdx.x, red);
}

// ------------------------------------------------------------------ dV = P^T dO, dK = dS^T Q
// Workgroup = 4 waves = 128 keys of one (batch, head), wave = 32 keys (one block column); row tiles of 32.  Q and
// dO rows and the wave's P and dS blocks pass through LDS, everything is read with transpose reads (the contraction
// runs over the rows); k slots of a lane group: rows 8g, 8g+2, 8g+4, 8g+6, then the odd ones, which is how
// the blocks keep them.  Loads are one row tile ahead in registers.
constexpr int KV_WAVES = 4;
template <int D> struct KvLds {
    static constexpr int RST = D * 2 + 16;            // bytes per staged row
    static constexpr int rows = 32 * RST;             // one matrix, [parity][16 row pairs]
    static constexpr int blocks = KV_WAVES * 2 * SC_BLK * 2;
    static constexpr int buf = 2 * rows + blocks;
    static constexpr int total = 2 * buf;
};

template <int D, typename TO>
__device__ __forceinline__ void dkdv_tile(int B, int H, int N, int causal, int n_rt, int n_kt, const bf16_t *__restrict__ Q,
                                          const bf16_t *__restrict__ dO, const bf16_t *__restrict__ Pws,
                                          const bf16_t *__restrict__ dSws, TO *__restrict__ dK, TO *__restrict__ dV, int h, int b,
                                          int z, unsigned char *smem) {
    using Lds = KvLds<D>;
    constexpr int DB = D / 16, CPR = D / 8, LD = 32 * CPR / (KV_WAVES * 64) > 0 ? 32 * CPR / (KV_WAVES * 64) : 1;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int kt = z * KV_WAVES + wave;          // this wave's block column
    const size_t bh = (size_t)b * H + h;
    const bf16_t *Qb = Q + bh * N * D, *Ob = dO + bh * N * D;
    const size_t wso = (size_t)b * chain_ds_block_off(causal != 0, n_rt, n_kt) * H + h;   // blocks lie [batch][block][head]
    const int kt_c = min(kt, n_rt - 1);                   // (N keys and N rows: n_rt columns exist)
    const bool own = kt < n_rt;
    const size_t col = wso + (chain_ds_block_off(causal != 0, n_rt, kt_c) - chain_ds_first_rt(causal != 0, kt_c)) * H;
    const int rt0 = causal ? z * KV_WAVES : 0;

    f32x4 acc_v[2][DB], acc_k[2][DB];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc_v[kb][db] = acc_k[kb][db] = (f32x4){0.f, 0.f, 0.f, 0.f};

    u32x4 qr[LD], orr[LD], pr[2], sr[2];
    auto load = [&](int rt) {
#pragma unroll
        for (int i = 0; i < LD; ++i) {
            const int c = (tid + i * KV_WAVES * 64) % (32 * CPR), row = min(rt * 32 + c / CPR, N - 1), cc = c % CPR;
            qr[i] = *reinterpret_cast<const u32x4 *>(Qb + (size_t)row * D + cc * 8);
            orr[i] = *reinterpret_cast<const u32x4 *>(Ob + (size_t)row * D + cc * 8);
        }
        // (columns start at row tile kt under the causal mask: an earlier one is not read)
        const size_t o = (col + (size_t)max(rt, causal ? kt_c : 0) * H) * SC_BLK + lane * 8;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            pr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(Pws + o + i * 512));
            sr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(dSws + o + i * 512));
        }
    };
    // From the last row tile up: blocks of keys that start together then read the same rows of Q and dO at the same time, whatever
    // their lengths under the causal mask (2.64 GB read instead of 2.98, of which 2.28 are needed, and the memory is what bounds
    // this).  us, from the first row tile down and from the last one up: B4 H16 N4096 d128 494 -> 447, B2 H32 N2048 d64 120 -> 115, B4 H16 N2048 d64
    // 123 -> 115, with dQ in one launch B2 H32 N1024 d128 83 -> 77.
    load(n_rt - 1);
    for (int rt = n_rt - 1; rt >= rt0; --rt) {
        unsigned char *buf = smem + (rt & 1) * Lds::buf;
        unsigned char *Ql = buf, *Ol = buf + Lds::rows, *Pl = buf + 2 * Lds::rows + wave * 2 * SC_BLK * 2, *Sl = Pl + SC_BLK * 2;
#pragma unroll
        for (int i = 0; i < LD; ++i) {
            const int c = tid + i * KV_WAVES * 64, row = c / CPR, cc = c % CPR;
            if (c < 32 * CPR) {
                // (rows past the last: copies of the last one, which P = dS = 0 takes out)
                const int o = ((row & 1) * 16 + (row >> 1)) * Lds::RST + cc * 16;
                *reinterpret_cast<u32x4 *>(Ql + o) = qr[i];
                *reinterpret_cast<u32x4 *>(Ol + o) = orr[i];
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<u32x4 *>(Pl + lane * 16 + i * 1024) = pr[i];
            *reinterpret_cast<u32x4 *>(Sl + lane * 16 + i * 1024) = sr[i];
        }
        lds_barrier();
        if (rt > rt0) load(rt - 1);
        if (!own || (causal && rt < kt)) continue;
        bf16x8 pf[2], sf[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            // block element [parity][key half kb][pair][16 keys]: pairs 4g .. 4g+3 of both parities
            const bf16x4 pl = lds_read_tr4x16(Pl + kb * 512, 32, 4 * g, 0, n), ph = lds_read_tr4x16(Pl + 1024 + kb * 512, 32, 4 * g, 0, n);
            const bf16x4 sl = lds_read_tr4x16(Sl + kb * 512, 32, 4 * g, 0, n), sh = lds_read_tr4x16(Sl + 1024 + kb * 512, 32, 4 * g, 0, n);
            pf[kb] = __builtin_shufflevector(pl, ph, 0, 1, 2, 3, 4, 5, 6, 7);
            sf[kb] = __builtin_shufflevector(sl, sh, 0, 1, 2, 3, 4, 5, 6, 7);
        }
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const bf16x4 ol = lds_read_tr4x16(Ol, Lds::RST, 4 * g, db * 16, n), oh = lds_read_tr4x16(Ol + 16 * Lds::RST, Lds::RST, 4 * g, db * 16, n);
            const bf16x4 ql = lds_read_tr4x16(Ql, Lds::RST, 4 * g, db * 16, n), qh = lds_read_tr4x16(Ql + 16 * Lds::RST, Lds::RST, 4 * g, db * 16, n);
            const bf16x8 of = __builtin_shufflevector(ol, oh, 0, 1, 2, 3, 4, 5, 6, 7), qf = __builtin_shufflevector(ql, qh, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                // rows of the product = head-dim columns, so that a lane holds four consecutive ones of a key
                acc_v[kb][db] = mfma_bf16(of, pf[kb], acc_v[kb][db]);
                acc_k[kb][db] = mfma_bf16(qf, sf[kb], acc_k[kb][db]);
            }
        }
    }
    if (!own) return;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        const int key = kt * 32 + kb * 16 + n;
        if (key >= N) continue;
        const size_t o = (bh * N + key) * D + 4 * g;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if constexpr (sizeof(TO) == 2) {
                bf16x4 v, k;
#pragma unroll
                for (int r = 0; r < 4; ++r) { v[r] = (bf16_t)acc_v[kb][db][r]; k[r] = (bf16_t)acc_k[kb][db][r]; }
                *reinterpret_cast<bf16x4 *>(dV + o + 16 * db) = v;
                *reinterpret_cast<bf16x4 *>(dK + o + 16 * db) = k;
            } else {
                *reinterpret_cast<f32x4 *>(dV + o + 16 * db) = acc_v[kb][db];
                *reinterpret_cast<f32x4 *>(dK + o + 16 * db) = acc_k[kb][db];
            }
        }
    }
}

template <int D, typename TO>
__global__ __launch_bounds__(KV_WAVES * 64, 2) void headmix_dkdv_kernel(int B, int H, int N, int causal, int n_rt, int n_kt,
                                                                     const bf16_t *__restrict__ Q,
                                                                     const bf16_t *__restrict__ dO,
                                                                     const bf16_t *__restrict__ Pws,
                                                                     const bf16_t *__restrict__ dSws,
                                                                     TO *__restrict__ dK, TO *__restrict__ dV) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    dkdv_tile<D, TO>(B, H, N, causal, n_rt, n_kt, Q, dO, Pws, dSws, dK, dV, blockIdx.x, blockIdx.y, blockIdx.z, smem);
}

// What follows the score kernel, in one launch: workgroups for dK and dV, then for dQ, then for dw.  Problems whose dQ tiles
// share keys among the waves (small ones) are bound by launches: three of 3 us of host time and 2 us of GPU time become one.
template <int D, typename TO>
__global__ __launch_bounds__(KV_WAVES * 64, 2) void headmix_products_kernel(Problem p, int n_rt, int n_kt, const bf16_t *__restrict__ Q,
                                                                            const bf16_t *__restrict__ K, const bf16_t *__restrict__ dO,
                                                                            const bf16_t *__restrict__ Pws, const bf16_t *__restrict__ dSws,
                                                                            int n_part, const float *__restrict__ dw_part,
                                                                            TO *__restrict__ dQ, TO *__restrict__ dK,
                                                                            TO *__restrict__ dV, float *__restrict__ dW) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int BH = p.B * p.H, kv = BH * ((p.Nk + 127) / 128), i = blockIdx.x;
    if (i < kv) {
        const int bh = i % BH;
        dkdv_tile<D, TO>(p.B, p.H, p.Nk, p.causal, n_rt, n_kt, Q, dO, Pws, dSws, dK, dV, bh % p.H, bh / p.H, i / BH, smem);
    } else if (i < kv + BH * n_rt) {
        const int j = i - kv, bh = j % BH;
        dq_rows::tile<D, TO, true>(p, K, dSws, nullptr, n_kt, n_rt, 1, dQ, bh % p.H, bh / p.H, n_rt - 1 - j / BH, smem);
    } else {
        dw_sum(n_part, p.H * p.H, dw_part, dW, i - kv - BH * n_rt, reinterpret_cast<float (*)[17]>(smem));
    }
}

Plan score_plan(int B, int H, int N, int causal) {
    return H == 16 ? make_plan<ScoreTile<16, 32>>(B, N, causal) : make_plan<ScoreTile<32, 32>>(B, N, causal);
}
// Asking ahead pays where a workgroup has many steps: us without and with it, B4 N4096 (258 steps) 1231 / 1098, B4 N3700 (210)
// 995 / 974, B4 N3200 (158) 726 / 704, B8 N2048 (130) 626 / 576, B4 N2900 (131) 598 / 595; B3 N3300 (128) 562 / 564, B4 N2700 (114)
// 510 / 521, B3 N3000 (105) 463 / 470.  Without the mask the gain begins further up: B2 N4096 (256) 1092 / 1019, B2 N3600 (200)
// 881 / 836, B4 N2500 (195) 896 / 874; B8 N1750 (189) 789 / 804, B2 N3300 (169) 664 / 671, B2 N3000 (138) 565 / 570, B4 N2000 (124)
// 534 / 555.  d = 64, whose loads have more chunks in flight, and 32 heads, whose steps take longer, gain nothing.
bool score_ahead(const Problem &p, const Plan &plan) { return p.H == 16 && p.d == 128 && plan.share > (p.causal ? 128 : 192); }

// What precedes the score kernel, in one launch: K and V in fragment order, then D and LSE of the rows.
template <int D, typename TO>
__global__ __launch_bounds__(256) void headmix_prepare_kernel(int N, int n_t16, size_t n_frag, size_t rows, const bf16_t *__restrict__ K,
                                                              const bf16_t *__restrict__ V, const TO *__restrict__ O,
                                                              const bf16_t *__restrict__ dO, const float *__restrict__ M,
                                                              const float *__restrict__ L, bf16_t *__restrict__ KF,
                                                              bf16_t *__restrict__ VF, float *__restrict__ Dl, float *__restrict__ LSE) {
    const size_t first = (n_frag + 3) / 4;
    if (blockIdx.x < first) frag_order<D>((size_t)blockIdx.x * 4 + (threadIdx.x >> 6), N, n_t16, K, V, KF, VF, n_frag);
    else row_stats(blockIdx.x - first, rows, D, O, dO, M, L, Dl, LSE);
}
template <int D>
hipError_t launch_prepare(const Problem &p, int o_dt, const void *k, const void *v, const void *o, const void *d_o, const float *m,
                          const float *l, void *kf, void *vf, float *Dl, float *lse, hipStream_t s) {
    const size_t n_frag = frag_count(p.B * p.H, p.Nk, D), rows = (size_t)p.B * p.H * p.Nq;
    const unsigned grid = (unsigned)((n_frag + 3) / 4 + (rows + 15) / 16);
    const int n_t16 = chain_row_tiles(p) * 2;
#define CALL(TO)                                                                                                              \
    headmix_prepare_kernel<D, TO><<<grid, 256, 0, s>>>(p.Nk, n_t16, n_frag, rows, (const bf16_t *)k, (const bf16_t *)v, (const TO *)o, \
                                                       (const bf16_t *)d_o, m, l, (bf16_t *)kf, (bf16_t *)vf, Dl, lse)
    if (o_dt == CONVATTN_BF16) CALL(bf16_t);
    else CALL(float);
#undef CALL
    return hipGetLastError();
}

template <int H, int D, bool AHEAD = false>
hipError_t launch_scores(const ScoreArgs &a, hipStream_t s) {
    constexpr int lds = ScoreTile<H, D>::lds;
    static_assert(ScoreTile<H, D>::WAVES * ScoreTile<H, D>::ROOM <= ScoreTile<H, D>::w_off * 4, "w stays where the rows are turned");
    static_assert(lds <= 160 * 1024 && ScoreTile<H, D>::WAVES * H * H * 4 <= lds, "LDS budget");
    hipError_t e = set_max_lds_once<headmix_scores_kernel<H, D, AHEAD>>(lds);
    if (e != hipSuccess) return e;
    headmix_scores_kernel<H, D, AHEAD><<<plan_grid(a.plan), ScoreTile<H, D>::WAVES * 64, lds, s>>>(a);
    return hipGetLastError();
}

template <int D, typename TO>
hipError_t launch_dkdv(const Problem &p, const void *q, const void *d_o, const bf16_t *P, const bf16_t *dS, void *dk, void *dv,
                       hipStream_t s) {
    constexpr int lds = KvLds<D>::total;
    hipError_t e = set_max_lds_once<headmix_dkdv_kernel<D, TO>>(lds);
    if (e != hipSuccess) return e;
    headmix_dkdv_kernel<D, TO><<<dim3(p.H, p.B, (p.Nk + 127) / 128), KV_WAVES * 64, lds, s>>>(
        p.B, p.H, p.Nk, p.causal, chain_row_tiles(p), chain_key_tiles(p), (const bf16_t *)q, (const bf16_t *)d_o, P, dS, (TO *)dk, (TO *)dv);
    return hipGetLastError();
}

template <int D, typename TO>
hipError_t launch_products(const Problem &p, const ScoreArgs &a, const void *k, void *dq, void *dk, void *dv, float *dw, hipStream_t s) {
    constexpr int lds = KvLds<D>::total > dq_rows::lds_by_keys<D> ? KvLds<D>::total : dq_rows::lds_by_keys<D>;
    hipError_t e = set_max_lds_once<headmix_products_kernel<D, TO>>(lds);
    if (e != hipSuccess) return e;
    const int n_rt = chain_row_tiles(p), grid = p.B * p.H * ((p.Nk + 127) / 128 + n_rt) + p.H * p.H / 16;
    headmix_products_kernel<D, TO><<<grid, KV_WAVES * 64, lds, s>>>(p, n_rt, chain_key_tiles(p), a.Q, (const bf16_t *)k, a.dO, a.P, a.dS,
                                                                   a.plan.n_wg, a.dw_part, (TO *)dq, (TO *)dk, (TO *)dv, dw);
    return hipGetLastError();
}

}  // namespace

// K (or V) in fragment order
size_t headmix_frag_bytes(const Problem &p) { return (size_t)p.B * p.H * chain_row_tiles(p) * 32 * p.d * 2; }
int headmix_score_wgs(int B, int H, int N, int causal) { return score_plan(B, H, N, causal).n_wg; }

hipError_t headmix_bwd_fused(const Problem &p, int grad_dt, const void *q, const void *k, const void *v, const float *w,
                             int o_dt, const void *o, const void *d_o, const float *m, const float *l, float *lse, float *Dl, void *P,
                             void *dS, void *kv_frag, float *dw_part, void *dq, void *dk, void *dv, float *dw, hipStream_t s) {
    const Plan plan = score_plan(p.B, p.H, p.Nq, p.causal);
    const bool want_kv = dk != nullptr;
    const ScoreArgs a{p.B, p.Nq, p.causal, chain_row_tiles(p), chain_key_tiles(p), plan, p.scale,
                      (const bf16_t *)q, (const bf16_t *)kv_frag, (const bf16_t *)kv_frag + headmix_frag_bytes(p) / 2, (const bf16_t *)d_o, w, lse, Dl,
                      (bf16_t *)P, (bf16_t *)dS, dq ? dw_part : nullptr};
    void *kf = kv_frag, *vf = static_cast<unsigned char *>(kv_frag) + headmix_frag_bytes(p);
    hipError_t e = p.d == 32   ? launch_prepare<32>(p, o_dt, k, v, o, d_o, m, l, kf, vf, Dl, lse, s)
                   : p.d == 64 ? launch_prepare<64>(p, o_dt, k, v, o, d_o, m, l, kf, vf, Dl, lse, s)
                               : launch_prepare<128>(p, o_dt, k, v, o, d_o, m, l, kf, vf, Dl, lse, s);
    if (e != hipSuccess) return e;
    e = hipErrorInvalidValue;
    if (p.H == 16)
        e = p.d == 32              ? launch_scores<16, 32>(a, s)
            : p.d == 64            ? launch_scores<16, 64>(a, s)
            : score_ahead(p, plan) ? launch_scores<16, 128, true>(a, s)
                                   : launch_scores<16, 128>(a, s);
    if (p.H == 32) e = p.d == 32 ? launch_scores<32, 32>(a, s) : p.d == 64 ? launch_scores<32, 64>(a, s) : launch_scores<32, 128>(a, s);
    if (e != hipSuccess) return e;
    if (want_kv && dq && dq_rows::by_keys(p, true)) {
#define CALL(DD) (grad_dt == CONVATTN_BF16 ? launch_products<DD, bf16_t>(p, a, k, dq, dk, dv, dw, s) \
                                           : launch_products<DD, float>(p, a, k, dq, dk, dv, dw, s))
        return p.d == 32 ? CALL(32) : p.d == 64 ? CALL(64) : CALL(128);
#undef CALL
    }
    if (want_kv) {
#define CALL(DD) (grad_dt == CONVATTN_BF16 ? launch_dkdv<DD, bf16_t>(p, q, d_o, a.P, a.dS, dk, dv, s) \
                                           : launch_dkdv<DD, float>(p, q, d_o, a.P, a.dS, dk, dv, s))
        e = p.d == 32 ? CALL(32) : p.d == 64 ? CALL(64) : CALL(128);
#undef CALL
        if (e != hipSuccess) return e;
    }
    if (dq) {
        e = mfma_dq_from_rows(p, grad_dt, k, dS, nullptr, dq, s, true);
        if (e != hipSuccess) return e;
        headmix_dw_sum_kernel<<<p.H * p.H / 16, 256, 0, s>>>(plan.n_wg, p.H * p.H, dw_part, dw);
        e = hipGetLastError();
    }
    return e;
}

}  // namespace convattn
