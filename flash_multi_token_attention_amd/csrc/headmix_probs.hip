// Forward of head-mixing attention (gfx950): O_h = softmax(scale sum_h' w[h][h'] Q_h' K_h'^T + causal mask) V_h.
//
// The head mix couples all heads of a (row, key) pair, the product with V all keys of a head.  In one workgroup, O of
// all heads (H d floats per row) and the Q fragments leave the registers no room for anything to be loaded
// ahead (measured at B4 H16 N4096 d128: 1.9 ms with 40 registers spilled, the 16-row form before it 1.8 ms).
// So the pass is cut there: headmix_probs_kernel writes the probabilities as bf16 blocks (the operand precision of the
// product), un-normalised, and headmix_pv_kernel multiplies them with V and divides by the row sums.
//
// The probabilities of a row's 32 keys in a block are exp2(z - m) with m the largest score of these keys, so that the
// largest of them is exactly 1: that element is what the rounding to bf16 costs most.  Errors of O against 64 bits, relative
// to its norm (rounding O itself is 1.6e-3): 1.87 to 2.01e-3 over N = 201 to 2048, d = 32 to 128, 16 and 32 heads; with one reference for
// all keys of a row 2.06 to 2.34e-3, with a running maximum per row 1.89 to 2.22e-3.  m is kept per (block, head, row), 1/16
// of the blocks' bytes; the product scales each block's contribution by exp2(m - M), M the row's largest score.  This costs the
// call 1 to 3 % beside one reference per row.  A segment of a row's keys sums its probabilities relative to a reference of
// its own, the largest score of its first block, moved where a score exceeds it by more than kSlack; the product kernel
// puts the segments together.
#include "headmix_common.hpp"

namespace convattn {
namespace {

using namespace headmix;

constexpr float kSlack = 60.f;      // log2 units: sums of terms of 2^60 stay far inside fp32
constexpr float kFloor = -126.f;    // blocks whose scores are all below this, relative to the reference, are zeros

// 16 heads: 16 waves of 128 registers (one head each), 32 rows x 32 keys per step; 32 heads: 8 waves of 256
// registers, 16 rows x 32 keys.  Two score buffers: the products of a step run under the mix of the step before it,
// one barrier per step.
template <int H, int D> struct ProbTile : Tile<H, H == 16 ? 16 : 8, H == 16 ? 32 : 16> {
    using B = Tile<H, H == 16 ? 16 : 8, H == 16 ? 32 : 16>;
    static constexpr int ROOM = B::R * (D * 2 + 16);        // a head's rows while they are turned
    static constexpr int w_off = 2 * B::arr * 4 > B::WAVES * ROOM ? 2 * B::arr : B::WAVES * ROOM / 4, sp_off = w_off + H * B::WST,
                         lds = sp_off * 4 + (H == 32 ? kSplitBytes : 0);   // (H = 32: the split of w behind it)
};

struct ProbArgs {
    int B, N, causal, n_rt32, n_kt;
    Plan plan;
    float scale;
    const bf16_t *Q, *KF;    // KF: fragment order
    const float *W;
    bf16_t *P;               // blocks
    float *top;              // largest score (log2 units) of a row in a block [B][block][H][32 rows]
    float *stats;            // [B][segment][reference, largest score, sum][H][N]
};

template <int H, int D>
__global__ __launch_bounds__((ProbTile<H, D>::WAVES * 64)) void headmix_probs_kernel(ProbArgs a) {
    using T = ProbTile<H, D>;
    constexpr int RB = T::RB, R = T::R, KT = T::KT, KB = T::KB, RW = T::RW, HS = T::HS, HPW = T::HPW, HB = T::HB,
                  KS = D / 32, NCH = HPW * KB;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    float *lds = reinterpret_cast<float *>(smem);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane_id = threadIdx.x & 63;
    const int id = share_of_workgroup(a.plan), N = a.N, h0 = wave * HPW;
    if (id < 0) return;
    for (int i = threadIdx.x; i < H * H; i += T::WAVES * 64) {
        const float w = a.W[i] * (a.scale * kLog2e);
        lds[T::w_off + (i / H) * T::WST + i % H] = w;
        if constexpr (H == 32) put_split(lds + T::sp_off, i / H, i % H, w);
    }
    for (int x_pos = id * a.plan.share, x_end = (int)min((long long)x_pos + a.plan.share, (long long)a.B * a.plan.entry_len); x_pos < x_end;) {
    const Segment sg = find_segment(a.plan, id, x_pos, false);
    const int b = sg.b, rt = sg.rt, n_steps = sg.len();
    x_pos += n_steps;
    const int segment = __builtin_amdgcn_readfirstlane(id - a.plan.start(b, rt) / a.plan.share);
    int lane = lane_id;
    asm volatile("" : "+v"(lane));   // (no registers for what could be kept from segment to segment)
    const int g = lane >> 4, n = lane & 15, i0 = rt * R;

    bf16x8 qf[HPW][RB][KS];
    {
#pragma unroll
        for (int t = 0; t < HPW; ++t)
            turn_rows<T, D>(qf[t], a.Q + ((size_t)b * H + h0 + t) * N * D, i0, N, smem + wave * T::ROOM);
        lds_barrier();
    }
    const float *wf_l = lds + T::w_off + n * T::WST + 4 * g;

    // ---- score phase: chunks of one head and 16 keys, K rows two chunks ahead ----
    bf16x8 kf[2][KS];
    const int n_t16 = a.n_rt32 * 2;
    auto load_chunk = [&](int step, int c) {
        const bf16_t *kp = a.KF + (((size_t)b * H + h0 + c / KB) * n_t16 + step * KB + c % KB) * KS * 512;   // (uniform)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kf[c & 1][ks] = *reinterpret_cast<const bf16x8 *>(kp + lane * 8 + ks * 512);
    };
    auto score_chunk = [&](float *S, int c) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) s = mfma_bf16(kf[c & 1][ks], qf[c / KB][rb][ks], s);
            *reinterpret_cast<f32x4 *>(S + (h0 + c / KB) * HS + (rb * 16 + n) * KT + 4 * T::slot(rb * 16 + n, 4 * (c % KB) + g)) = s;
        }
    };
    // all chunks of `step` into S, loading the first two of step `next`
    auto scores = [&](float *S, int step, int next) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            score_chunk(S, c);
            if (c + 2 < NCH) load_chunk(step, c + 2);
            else load_chunk(next, c + 2 - NCH);
        }
    };

    // ---- mixing phase: lane (g, n) = heads 16x + 4g .. +3, tile row lr, keys 4q4 .. 4q4+3 ----
    const int lr = wave * RW + (n & (RW - 1)), q4 = n / RW, row = T::row(i0, lr), brow = row & 31;
    const int pos = lr * KT + 4 * T::slot(lr, q4);
    f32x4 nref[HB], top[HB], l_sum[HB];   // negative reference; largest score, relative to the reference
#pragma unroll
    for (int x = 0; x < HB; ++x) {
        nref[x] = l_sum[x] = (f32x4){0.f, 0.f, 0.f, 0.f};
        top[x] = (f32x4){kNegInf, kNegInf, kNegInf, kNegInf};
    }
    // (z starts at from[]: the negative references of the lane's row)
    auto mix = [&](f32x4 (&z)[HB][4], const f32x4 (&from)[HB], const float *S, int step) {
        auto start = [&] {
#pragma unroll
            for (int x = 0; x < HB; ++x)
#pragma unroll
                for (int t = 0; t < 4; ++t) z[x][t] = from[x];
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
        if ((a.causal && step * KT + KT - 1 > i0) || step * KT + KT > N) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int key = step * KT + 4 * q4 + t;
                if (key >= N || (a.causal && key > row)) {
#pragma unroll
                    for (int x = 0; x < HB; ++x) z[x][t] = (f32x4){kNegInf, kNegInf, kNegInf, kNegInf};
                }
            }
        }
    };
    auto row_max = [&](float v) {   // over the lanes of a row
        v = fmaxf(v, row16_rot<8>(v));
        v = fmaxf(v, row16_rot<4>(v));
        if constexpr (RW == 2) v = fmaxf(v, row16_rot<2>(v));
        return v;
    };
    const long long n_blk = chain_ds_block_off(a.causal != 0, a.n_rt32, a.n_kt);
    const int out = (((brow & 1) * 2 + ((4 * q4) >> 4)) * 16 + (brow >> 1)) * 16 + ((4 * q4) & 15) + 4 * g * kBlock;
    static_assert(KT == 32, "a step is a column of blocks");

    auto probs = [&](const float *S, int u) {
        const int step = sg.step(u);
        f32x4 z[HB][4], bm[HB];   // bm: largest score of the row's keys in this block
        mix(z, nref, S, step);
        bool move = u == 0;
#pragma unroll
        for (int x = 0; x < HB; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                bm[x][r] = row_max(fmaxf(fmaxf(z[x][0][r], z[x][1][r]), fmaxf(z[x][2][r], z[x][3][r])));
                move |= bm[x][r] > kSlack;
            }
        if (__any(move)) {   // the first block of the segment; rare after it
#pragma unroll
            for (int x = 0; x < HB; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float up = u == 0 ? (bm[x][r] > kNegInf ? bm[x][r] : 0.f) : fmaxf(0.f, bm[x][r]);
                    l_sum[x][r] = u == 0 ? 0.f : l_sum[x][r] * fast_exp2(-up);
                    nref[x][r] -= up;
                    top[x][r] -= up;
                    bm[x][r] -= up;
#pragma unroll
                    for (int t = 0; t < 4; ++t) z[x][t][r] -= up;
                }
        }
        const int kt = step;
        const size_t blk = (size_t)b * n_blk + chain_ds_block_off(a.causal != 0, a.n_rt32, kt) + i0 / 32 - chain_ds_first_rt(a.causal != 0, kt);
        bf16_t *p_out = a.P + blk * H * kBlock;
        float *t_out = a.top + (blk * H + 4 * g) * 32 + brow;
#pragma unroll
        for (int x = 0; x < HB; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float m = fmaxf(bm[x][r], kFloor), f = fast_exp2(-m);
                bf16x4 pb;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float p = fast_exp2(z[x][t][r]);
                    l_sum[x][r] += p;
                    pb[t] = (bf16_t)(p * f);
                }
                top[x][r] = fmaxf(top[x][r], m);
                __builtin_nontemporal_store(__builtin_bit_cast(u32x2, pb), reinterpret_cast<u32x2 *>(p_out + out + (16 * x + r) * kBlock));
                if (q4 == 0) t_out[(16 * x + r) * 32] = m - nref[x][r];
            }
    };

    float *buf0 = lds, *buf1 = lds + T::arr;
    const auto later = [&](int i) { return sg.step(min(i, n_steps - 1)); };
    load_chunk(sg.step(0), 0);
    load_chunk(sg.step(0), 1);
    scores(buf0, sg.step(0), later(1));
    lds_barrier();
    for (int u = 0; u < n_steps; ++u) {
        float *cur = u & 1 ? buf1 : buf0, *nxt = u & 1 ? buf0 : buf1;
        // (half of the waves take the scores of the next step first, half the mix of this one: one half's LDS and vector work
        // runs under the other's products)
        const bool first = wave < T::WAVES / 2, more = u + 1 < n_steps;
        const int next = later(u + 1), ahead = later(u + 2);
        if (more && first) scores(nxt, next, ahead);
        probs(cur, u);
        if (more && !first) scores(nxt, next, ahead);
        lds_barrier();
    }

    float *st = a.stats + ((size_t)b * a.plan.max_segments + segment) * 3 * H * N;
#pragma unroll
    for (int x = 0; x < HB; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float l = l_sum[x][r];
            l += row16_rot<8>(l);
            l += row16_rot<4>(l);
            if constexpr (RW == 2) l += row16_rot<2>(l);
            const size_t o = (size_t)(16 * x + 4 * g + r) * N + row, hn = (size_t)H * N;
            if (q4 == 0 && row < N) {
                st[o] = -nref[x][r];
                st[hn + o] = top[x][r] - nref[x][r];
                st[2 * hn + o] = l;
            }
        }
    }   // segments
}

// O = P V / (sum of P): the product kernel of dQ = dS K (bwd_dq_rows.hip) with the row sums, L and M at the end.
// Workgroup = 4 waves = 128 rows of one (batch, head), wave = 32 rows, steps of 64 keys; P blocks go straight
// into the operand registers (non-temporal), V passes through LDS.  Each block's product starts at zero and is added with the
// rows' factors: four fp32 operations per lane to each matrix instruction, beside the reads of P that bound the kernel
// (B4 H16 N4096 d128: 1.07 GB of P and 0.07 GB of largest scores, 0.25 ms = 4.6 TB/s; without the factors 0.22 ms; B2 H32
// N2048 d64 61 us as without them; B1 H16 N4096 d32 69 us, without 58).  What is loaded ahead and what the scheduler may
// mix are held down, or it takes registers for the products of many column blocks at once and fewer waves are there to wait
// for memory: d = 128 one step ahead and 3 waves per SIMD (two steps, 2 waves: 0.32 ms, with the barriers between
// column blocks 0.27; two steps, 3 waves: 16 to 24 registers spilled, 0.36 to 0.40); d <= 64 two steps ahead (one: 66 and
// 73 us).
constexpr int PV_WAVES = 4, PV_ROWS = 128, PV_KEYS = 64;

template <int D, typename TO>
__global__ __launch_bounds__(PV_WAVES * 64, 3) void headmix_pv_kernel(ProbArgs a, int H, const bf16_t *__restrict__ V,
                                                                   TO *__restrict__ O, float *__restrict__ L, float *__restrict__ M) {
    constexpr int RST = D * 2 + 16, DB = D / 16, CPR = D / 8, LD = PV_KEYS * CPR / (PV_WAVES * 64),
                  AHEAD = D == 128 ? 1 : 2, GROUP = D == 128 ? 2 : 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * PV_KEYS * RST];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int h = blockIdx.x, b = blockIdx.y, qt = gridDim.z - 1 - blockIdx.z;   // longest (causal) tiles first
    const int N = a.N, i0 = qt * PV_ROWS, rw = i0 + wave * 32, rt = rw / 32, n_rt = a.n_rt32;
    const bool causal = a.causal != 0, row_ok = rt < n_rt;
    const size_t bh = (size_t)b * H + h;
    const bf16_t *Vb = V + bh * N * D;
    const bf16_t *ws = a.P + ((size_t)b * chain_ds_block_off(causal, n_rt, a.n_kt) * H + h) * kBlock;

    // ---- the rows' statistics over the segments of their keys: lane n of block ob = row 2n + ob ----
    const int tile = (min(rt, n_rt - 1) << a.plan.split_shift) + (a.plan.split_shift ? n >> 3 : 0);   // the rows' tile
    const int t_start = a.plan.start(b, tile), t_first = t_start / a.plan.share;
    const int n_ch = (t_start + a.plan.len(tile) - 1) / a.plan.share - t_first + 1;
    float largest[2], inv[2];
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
        const int row = min(rw + 2 * n + ob, N - 1);
        const size_t hn = (size_t)H * N;
        const float *st = a.stats + (size_t)b * a.plan.max_segments * 3 * hn + (size_t)h * N + row;
        float r = st[0], m = st[hn], l = st[2 * hn];
        for (int c = 1; c < n_ch; ++c) {
            const float *s = st + (size_t)c * 3 * hn;
            const float rc = s[0], rn = fmaxf(r, rc);
            m = fmaxf(m, s[hn]);
            l = l * fast_exp2(r - rn) + s[2 * hn] * fast_exp2(rc - rn);
            r = rn;
        }
        l *= fast_exp2(r - m);
        largest[ob] = m;
        inv[ob] = 1.f / l;
        if (g == 0 && rw + 2 * n + ob < N) {
            M[bh * N + row] = m * (1.f / kLog2e);
            L[bh * N + row] = l;
        }
    }
    f32x4 acc[2][DB];
#pragma unroll
    for (int ob = 0; ob < 2; ++ob)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[ob][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int k_end = causal ? min(N, i0 + PV_ROWS) : N, n_steps = (k_end + PV_KEYS - 1) / PV_KEYS;
    struct Blocks { u32x4 p[2][2]; float2 top[2]; };   // [key half of the step]: probabilities of both row parities; largest scores
    u32x4 vr[LD];
    Blocks pr[AHEAD];
    const float *tops = a.top + ((size_t)b * chain_ds_block_off(causal, n_rt, a.n_kt) * H + h) * 32 + 2 * n;
    auto load_v = [&](int s) {
#pragma unroll
        for (int i = 0; i < LD; ++i) {
            const int c = tid + i * PV_WAVES * 64;
            vr[i] = load_row16_clamped<D>(Vb, s * PV_KEYS + c / CPR, N, (c % CPR) * 8);
        }
    };
    auto load_p = [&](int s, Blocks &pr) {
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
            const int kt = s * 2 + kp;
            // (a block that does not exist: any block that does; the registers are cleared before their use)
            const int rt_c = min(rt, n_rt - 1), kt_c = min(kt, causal ? rt_c : n_rt - 1);
            const size_t blk = (size_t)chain_ds_block_off(causal, n_rt, kt_c) + rt_c - chain_ds_first_rt(causal, kt_c);
            pr.top[kp] = *reinterpret_cast<const float2 *>(tops + blk * H * 32);
#pragma unroll
            for (int ob = 0; ob < 2; ++ob)
                pr.p[kp][ob] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(
                    ws + blk * H * kBlock + ((ob * 2 + (g >> 1)) * 16 + n) * 16 + 8 * (g & 1)));
        }
    };
    auto run_step = [&](int s, Blocks &pr) {
        unsigned char *Vs = smem + (s & 1) * PV_KEYS * RST;
#pragma unroll
        for (int i = 0; i < LD; ++i) {
            const int c = tid + i * PV_WAVES * 64;
            *reinterpret_cast<u32x4 *>(Vs + (c / CPR) * RST + (c % CPR) * 16) = zero_unless(s * PV_KEYS + c / CPR < N, vr[i]);
        }
        bf16x8 pf[2][2];
        float f[2][2];
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
            const int kt = s * 2 + kp;
            const bool ok = row_ok && kt < n_rt && (!causal || kt <= rt);
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) {
                pf[kp][ob] = __builtin_bit_cast(bf16x8, zero_unless(ok, pr.p[kp][ob]));
                f[kp][ob] = fast_exp2((ob ? pr.top[kp].y : pr.top[kp].x) - largest[ob]);
            }
        }
        __syncthreads();
        load_v(s + 1);
        load_p(s + AHEAD, pr);
        if (causal && s * PV_KEYS > rw + 31) return;  // every key of the step is after the wave's rows
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                if (db % GROUP == 0) __builtin_amdgcn_sched_barrier(0);
                const bf16x4 lo = lds_read_tr4x16(Vs, RST, kp * 32 + 8 * g, db * 16, n), hi = lds_read_tr4x16(Vs, RST, kp * 32 + 8 * g + 4, db * 16, n);
                const bf16x8 vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int ob = 0; ob < 2; ++ob) {
                    const f32x4 one = mfma_bf16(vf, pf[kp][ob], (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[ob][db][r] = fmaf(one[r], f[kp][ob], acc[ob][db][r]);
                }
            }
    };
    load_v(0);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) load_p(i, pr[i]);
    for (int s = 0; s < n_steps; s += AHEAD)
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (s + i < n_steps) run_step(s + i, pr[i]);
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
        const int row = rw + 2 * n + ob;
        if (row >= N) continue;
        TO *o = O + (bh * N + row) * D + 4 * g;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const f32x4 v = acc[ob][db] * inv[ob];
            if constexpr (sizeof(TO) == 2) {
                bf16x4 ov;
#pragma unroll
                for (int r = 0; r < 4; ++r) ov[r] = (bf16_t)v[r];
                *reinterpret_cast<bf16x4 *>(o + 16 * db) = ov;
            } else {
                *reinterpret_cast<f32x4 *>(o + 16 * db) = v;
            }
        }
    }
}

Plan prob_plan(const Problem &p) {
    return p.H == 16 ? make_plan<ProbTile<16, 32>>(p.B, p.Nq, p.causal) : make_plan<ProbTile<32, 32>>(p.B, p.Nq, p.causal);
}

template <int D>
__global__ __launch_bounds__(256) void frag_order_kernel(int N, int n_t16, const bf16_t *__restrict__ K, bf16_t *__restrict__ KF,
                                                         size_t n_frag) {
    frag_order<D>((size_t)blockIdx.x * 4 + (threadIdx.x >> 6), N, n_t16, K, nullptr, KF, nullptr, n_frag);
}

template <int H, int D, typename TO>
hipError_t launch(const Problem &p, const ProbArgs &a, const void *k, const void *v, void *o, float *l, float *m, hipStream_t s) {
    using T = ProbTile<H, D>;
    static_assert(T::lds <= 160 * 1024, "LDS budget");
    const size_t n_frag = frag_count(p.B * H, a.N, D);
    frag_order_kernel<D><<<(unsigned)((n_frag + 3) / 4), 256, 0, s>>>(a.N, a.n_rt32 * 2, (const bf16_t *)k, const_cast<bf16_t *>(a.KF), n_frag);
    hipError_t e = set_max_lds_once<headmix_probs_kernel<H, D>>(T::lds);
    if (e != hipSuccess) return e;
    headmix_probs_kernel<H, D><<<plan_grid(a.plan), T::WAVES * 64, T::lds, s>>>(a);
    headmix_pv_kernel<D, TO><<<dim3(H, p.B, (a.N + PV_ROWS - 1) / PV_ROWS), PV_WAVES * 64, 0, s>>>(a, H, (const bf16_t *)v, (TO *)o, l, m);
    return hipGetLastError();
}

}  // namespace

// K in fragment order, statistics of the segments, largest scores of the blocks, blocks
static size_t prob_stats_bytes(const Problem &p) { return ((size_t)p.B * prob_plan(p).max_segments * 3 * p.H * p.Nq * sizeof(float) + 255) / 256 * 256; }
static size_t prob_top_bytes(const Problem &p) { return chain_ds_bytes(p) / (kBlock * 2) * 32 * sizeof(float); }
size_t headmix_fwd_workspace(const Problem &p) { return headmix_frag_bytes(p) + prob_stats_bytes(p) + prob_top_bytes(p) + chain_ds_bytes(p); }

hipError_t headmix_fwd_blocks(const Problem &p, int out_dt, const void *q, const void *k, const void *v, const float *w,
                              void *ws, void *o, float *l, float *m, hipStream_t s) {
    unsigned char *base = static_cast<unsigned char *>(ws);
    const size_t fb = headmix_frag_bytes(p), sb = prob_stats_bytes(p), tb = prob_top_bytes(p);
    const ProbArgs a{p.B, p.Nq, p.causal, chain_row_tiles(p), chain_key_tiles(p), prob_plan(p), p.scale, (const bf16_t *)q,
                     (const bf16_t *)base, w, (bf16_t *)(base + fb + sb + tb), (float *)(base + fb + sb), (float *)(base + fb)};
#define CALL(HH, DD) (out_dt == CONVATTN_BF16 ? launch<HH, DD, bf16_t>(p, a, k, v, o, l, m, s) : launch<HH, DD, float>(p, a, k, v, o, l, m, s))
    if (p.H == 16) return p.d == 32 ? CALL(16, 32) : p.d == 64 ? CALL(16, 64) : CALL(16, 128);
    if (p.H == 32) return p.d == 32 ? CALL(32, 32) : p.d == 64 ? CALL(32, 64) : CALL(32, 128);
#undef CALL
    return hipErrorInvalidValue;
}

}  // namespace convattn
