// Small bandwidth-bound helpers around the conv-attention kernels:
// backward preparation (D, LSE), the ordered dW reduction and the decode
// split merge.
#include "reduce_common.hpp"

namespace convattn {
namespace {

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void preprocess_kernel(size_t rows, int d, const TO *__restrict__ O,
                                                         const TI *__restrict__ dO,
                                                         const float *__restrict__ M,
                                                         const float *__restrict__ L,
                                                         float *__restrict__ D, float *__restrict__ LSE) {
    row_stats(blockIdx.x, rows, d, O, dO, M, L, D, LSE);
}

// D, LSE and the dC scale of the bf16 backward from one reading of O, dO and V: D / 8 lanes per row, x = rows of one of
// `chunks` parts of a (batch, head).  One part: the workgroup has the maxima of all of them and writes the scale;
// several: it leaves its maxima (the layout of dc_scale_partial_kernel) for dc_scale_finish.
template <int D, typename TO>
__global__ void bwd_prepare_kernel(int Nq, int Nk, const TO *__restrict__ O, const bf16_t *__restrict__ dO,
                                   const bf16_t *__restrict__ V, const float *__restrict__ M, const float *__restrict__ L,
                                   float *__restrict__ Dl, float *__restrict__ LSE, float *__restrict__ part,
                                   float *__restrict__ scale) {
    constexpr int LPR = D / 8;
    __shared__ float red[2][16];
    const size_t bh = (size_t)blockIdx.z * gridDim.y + blockIdx.y;   // y = head, z = batch
    const int tid = threadIdx.x, sub = tid % LPR, step = blockDim.x / LPR;
    float top[2] = {0.f, 0.f};
    auto bounds = [&](int n, int &lo, int &hi) {
        const int per = (n + gridDim.x - 1) / gridDim.x;
        lo = blockIdx.x * per;
        hi = min(n, lo + per);
    };
    int lo, hi;
    bounds(Nq, lo, hi);
    for (int r = lo + tid / LPR; r < hi; r += step) {
        const size_t row = bh * Nq + r;
        float o[8], g[8], s = 0.f;
        load8(O + row * D + sub * 8, o);
        load8(dO + row * D + sub * 8, g);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            s = fmaf(o[i], g[i], s);
            top[0] = fmaxf(top[0], fabsf(g[i]));
        }
#pragma unroll
        for (int m = LPR / 2; m >= 1; m >>= 1) s += __shfl_xor(s, m, LPR);
        if (sub == 0) {
            Dl[row] = s;
            LSE[row] = M[row] + __logf(L[row]);
        }
    }
    bounds(Nk, lo, hi);
    for (int r = lo + tid / LPR; r < hi; r += step) {
        float v[8];
        load8(V + (bh * Nk + r) * D + sub * 8, v);
#pragma unroll
        for (int i = 0; i < 8; ++i) top[1] = fmaxf(top[1], fabsf(v[i]));
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        top[x] = wave_max(top[x]);
        if ((tid & 63) == 0) red[x][tid >> 6] = top[x];
    }
    __syncthreads();
    if (tid < 2) {
        float mx = 0.f;
        for (int w = 0; w < (int)blockDim.x / 64; ++w) mx = fmaxf(mx, red[tid][w]);
        red[tid][0] = mx;
        if (gridDim.x > 1) part[(bh * gridDim.x + blockIdx.x) * 2 + tid] = mx;
    }
    if (gridDim.x > 1) return;
    __syncthreads();
    if (tid == 0) write_dc_scale(D, red[0][0], red[1][0], scale + 2 * bh);
}

__global__ __launch_bounds__(1024) void dw_reduce_kernel(int B, int H, int n_tiles, int ntap,
                                                         const float *__restrict__ part, float *__restrict__ dW) {
    __shared__ float red[kDwChains][64];
    dw_reduce_block<1024>(B, H, n_tiles, ntap, part, dW, blockIdx.x, blockIdx.y, red);
}

// x = 16-byte groups of a key block's dK, then dV, y = key block, z = (batch, head)
template <typename TO>
__global__ __launch_bounds__(256) void chain_reduce_kernel(Problem p, int share, int n_wg, const float *__restrict__ part,
                                                           TO *__restrict__ dK, TO *__restrict__ dV) {
    chain_reduce_block(p, share, n_wg, part, dK, dV, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Merge of up to MOST decode splits: one workgroup per (batch, head), one thread per output column.  A launch is as long as
// its loads take, so all of them are issued before the first is used.
template <int MOST, typename TO>
__global__ __launch_bounds__(128) void combine_few_kernel(int n_splits, int d, const float *__restrict__ O_part,
                                   const float *__restrict__ M_part, const float *__restrict__ L_part,
                                   TO *__restrict__ O, float *__restrict__ M, float *__restrict__ L) {
    const size_t bh = blockIdx.x;
    const float *mp = M_part + bh * n_splits;
    const float *lp = L_part + bh * n_splits;
    const int c = min((int)threadIdx.x, d - 1);   // (d <= 128)
    float ms[MOST], ls[MOST], os[MOST];
#pragma unroll
    for (int s = 0; s < MOST; ++s) {
        const int at = min(s, n_splits - 1);
        ms[s] = mp[at];
        ls[s] = lp[at];
        os[s] = O_part[(bh * n_splits + at) * d + c];
    }
    float m = kNegInf, l = 0.f, o = 0.f;
#pragma unroll
    for (int s = 0; s < MOST; ++s) m = fmaxf(m, ms[s]);
#pragma unroll
    for (int s = 0; s < MOST; ++s) {
        if (s >= n_splits || ms[s] == kNegInf) continue;
        const float f = __expf(ms[s] - m);
        l += ls[s] * f;
        o = fmaf(os[s], f, o);
    }
    if ((int)threadIdx.x < d) O[bh * d + c] = from_f32<TO>(o / l);
    if (threadIdx.x == 0) { M[bh] = m; L[bh] = l; }
}

// Merge of many decode splits: m = max m_s, l = sum l_s e^{m_s - m}, o = sum o_s e^{m_s - m} / l.
// A workgroup takes 32 output columns of one (batch, head).  All 256 threads scan the splits'
// (m_s, l_s) together (every workgroup of a head repeats this: at most 1024 pairs); for the
// outputs thread (g, c) adds the splits g, g+8, ... of column c, so a split's row is read with
// 128-byte loads and eight rows are in flight per pass, and the eight sums are added in order of g.
template <typename TO>
__global__ __launch_bounds__(256) void combine_kernel(int n_splits, int d, const float *__restrict__ O_part,
                                                      const float *__restrict__ M_part,
                                                      const float *__restrict__ L_part, TO *__restrict__ O,
                                                      float *__restrict__ M, float *__restrict__ L) {
    __shared__ float red_m[4], red_l[4], acc[8][32];
    const size_t bh = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *mp = M_part + bh * n_splits;
    const float *lp = L_part + bh * n_splits;
    float m = kNegInf;
    for (int s = tid; s < n_splits; s += 256) m = fmaxf(m, mp[s]);
#pragma unroll
    for (int x = 32; x >= 1; x >>= 1) m = fmaxf(m, __shfl_xor(m, x));
    if (lane == 0) red_m[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
    float l = 0.f;
    for (int s = tid; s < n_splits; s += 256) {
        const float ms = mp[s];
        if (ms != kNegInf) l = fmaf(lp[s], __expf(ms - m), l);
    }
#pragma unroll
    for (int x = 32; x >= 1; x >>= 1) l += __shfl_xor(l, x);
    if (lane == 0) red_l[wave] = l;
    __syncthreads();
    l = (red_l[0] + red_l[1]) + (red_l[2] + red_l[3]);

    const int c = tid & 31, g = tid >> 5, col = blockIdx.y * 32 + c;
    float o = 0.f;
    if (col < d) {
        const float *op = O_part + bh * n_splits * d + col;
#pragma unroll 4
        for (int s = g; s < n_splits; s += 8) {
            const float ms = mp[s];
            if (ms != kNegInf) o = fmaf(op[(size_t)s * d], __expf(ms - m), o);
        }
    }
    acc[g][c] = o;
    __syncthreads();
    if (tid < 32 && col < d) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += acc[i][c];
        O[bh * d + col] = from_f32<TO>(sum / l);
    }
    if (tid == 0 && blockIdx.y == 0) { M[bh] = m; L[bh] = l; }
}

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

}  // namespace

hipError_t bwd_preprocess(const Problem &p, int in_dt, int out_dt, const void *o, const void *d_o,
                          const float *m, const float *l, float *D, float *lse, hipStream_t s) {
    const size_t rows = (size_t)p.B * p.H * p.Nq;
    const unsigned grid = (unsigned)((rows + 15) / 16);
#define CALL(TI, TO) \
    preprocess_kernel<TI, TO><<<grid, 256, 0, s>>>(rows, p.d, (const TO *)o, (const TI *)d_o, m, l, D, lse)
    if (in_dt == CONVATTN_BF16 && out_dt == CONVATTN_BF16) CALL(bf16_t, bf16_t);
    else if (in_dt == CONVATTN_BF16) CALL(bf16_t, float);
    else if (out_dt == CONVATTN_BF16) CALL(float, bf16_t);
    else CALL(float, float);
#undef CALL
    return hipGetLastError();
}

// part: dc_scale as mfma_dc_scale leaves it ({s, log2 s} per (batch, head), then the maxima of kScaleChunks parts)
hipError_t bwd_prepare(const Problem &p, int out_dt, const void *o, const void *d_o, const void *v, const float *m, const float *l,
                       float *D, float *lse, float *dc_scale, hipStream_t s) {
    // (one workgroup reads 64 K elements of each tensor in about 4 us, as long as the second launch would take)
    const bool one = (long long)(p.Nq > p.Nk ? p.Nq : p.Nk) * p.d <= 65536;
    const dim3 grid(one ? 1 : kScaleChunks, p.H, p.B);
    float *part = dc_scale + (size_t)p.B * p.H * 2;
#define CALL(DD, TO)                                                                                                            \
    bwd_prepare_kernel<DD, TO><<<grid, one ? 1024 : 256, 0, s>>>(p.Nq, p.Nk, (const TO *)o, (const bf16_t *)d_o, (const bf16_t *)v, m, \
                                                                 l, D, lse, part, dc_scale)
#define PICK(DD) (out_dt == CONVATTN_BF16 ? CALL(DD, bf16_t) : CALL(DD, float))
    if (p.d == 32) PICK(32);
    else if (p.d == 64) PICK(64);
    else PICK(128);
#undef PICK
#undef CALL
    const hipError_t e = hipGetLastError();
    return e != hipSuccess || one ? e : dc_scale_finish(p, dc_scale, s);
}

hipError_t dw_reduce(const Problem &p, int n_tiles, const float *dw_part, float *dw, hipStream_t s) {
    dw_reduce_kernel<<<dim3(p.H, (p.c_q * p.c_k + 63) / 64), 1024, 0, s>>>(p.B, p.H, n_tiles, p.c_q * p.c_k, dw_part, dw);
    return hipGetLastError();
}

namespace {
// When the last workgroup of a launch ends: workgroups are handed to the CU that is free first, one at a time, in the order
// in which they are added.
class Schedule {
    float at_[256] = {0.f};   // CUs by the time they are free, ascending
    int cus_[256] = {256}, n_ = 1;

  public:
    void add(float cost, int wgs) {
        while (wgs > 0) {
            const int k = wgs < cus_[0] ? wgs : cus_[0];
            const float end = at_[0] + cost;
            wgs -= k;
            if ((cus_[0] -= k) == 0) {
                --n_;
                for (int i = 0; i < n_; ++i) { at_[i] = at_[i + 1]; cus_[i] = cus_[i + 1]; }
            }
            int i = n_;
            while (i > 0 && at_[i - 1] > end) --i;
            if (i > 0 && at_[i - 1] == end) { cus_[i - 1] += k; continue; }
            for (int r = n_++; r > i; --r) { at_[r] = at_[r - 1]; cus_[r] = cus_[r - 1]; }
            at_[i] = end;
            cus_[i] = k;
        }
    }
    float end() const { return at_[n_ - 1]; }
};
}  // namespace

// Row tiles per workgroup of the split backward, or 0: one workgroup per key block.  The launch is laid out on 256 CUs for each
// cut of the longest key block, from 1 1/4 to 8 parts; in units of a row tile a workgroup costs its tiles, 10 for set-up and wind-down and
// 1 more where its range ends inside the key block (windows of 7 to 11 query taps, whose tiles take longer: 4 and 1 up to d = 64, 6 and
// 2 at 128); what the reduction takes is in the margin over the unsplit launch.  The constants were fitted with one dense product per tap, against
// every cut for 2 to 64 heads of 640 to 8000 rows (482 shapes of 3x3 to 11x11 taps, d 32 to 128, a quarter of the last 221 not causal): 0.3 to
// 0.8 % over the best on average.  With two taps per product, 110 other such shapes: 1.7 % over the best of twelve cuts on average (unsplit
// 38 %), single ones up to 15 % (B1 H12 N2023 d32 7x7 105 us, into 1 3/4 parts 91), 8 of the 73 in parts 2 to 6 % slower than unsplit.
// (B2 H8 N1531 d64 11x11, us, whole backward without D: unsplit 133, into 3 parts 116, 1 1/2 parts 101; B1 H8 N2048 d64 7x7 137, 84, 100; with more
// than two rounds of workgroups a split loses: B1 H8 N8000 d128 6x11 771 us unsplit, 889 in 2 parts, B1 H12 N5000 486 and 563.)
// The limits: 12 to 19 row tiles would gain too (B1 H8 N512 d64 6x11 the whole backward 44 -> 30 us), which such calls, bound by
// the host (75 us for a step), show in a captured graph only.  Beyond 64 heads no cut gained (5 to 45 % slower at 80 to
// 256 heads of 640 to 4096 rows, dense products).  From 8192 rows on nothing is split, whatever the number of heads is, so that a head's results
// do not depend on how many others there are; up to four heads would gain (B1 H1 N16384 d128 1180 -> 632 us, B1 H4 N8192 614 -> 501),
// more would not (B1 H8 N8192 732 -> 749).
int chain_share(const Problem &p) {
    const int n_rt = chain_row_tiles(p), n_kb = mfma_kv_tiles(p);
    const long long heads = (long long)p.B * p.H;
    if (n_rt < 20 || p.Nq >= 8192 || heads > 64 || heads * n_kb > 1024) return 0;
    const bool wide = p.c_q > 6, small = p.d <= 64;
    const float fixed = !wide ? 10.f : small ? 4.f : 6.f, cut_end = wide && !small ? 2.f : 1.f, margin = wide ? 1.04f : 1.06f;
    const int n = (int)heads;
    float best = 0.f, none = 0.f;
    int share = 0;
    for (const int quarters : {4, 5, 6, 7, 8, 10, 12, 14, 16, 18, 20, 24, 28, 32}) {   // parts of the longest key block, in quarters
        const int s = quarters == 4 ? 0 : (4 * n_rt + quarters - 1) / quarters;
        if (quarters > 4 && s < 6) break;
        auto cost = [&](int kb, int parts) {
            const int len = chain_len(p, kb) > 0 ? chain_len(p, kb) : 0;
            return (float)len / parts + fixed + (parts > 1 ? cut_end : 0.f);
        };
        if (quarters > 4) {   // (no better than even shares, and than its longest workgroup)
            float sum = 0.f;
            for (int kb = 0; kb < n_kb; ++kb) sum += cost(kb, chain_parts(p, kb, s)) * chain_parts(p, kb, s);
            if (sum * n / 256.f >= best) continue;
        }
        Schedule launch;
        for (int kb = 0; kb < n_kb; ++kb) launch.add(cost(kb, chain_parts(p, kb, s)), n * chain_parts(p, kb, s));
        const float t = launch.end();
        if (quarters == 4) none = best = t;
        else if (margin * t < none && t < best) { best = t; share = s; }
    }
    return share;
}

hipError_t chain_reduce(const Problem &p, int out_dt, int share, const float *part, void *dk, void *dv, hipStream_t s) {
    const dim3 grid(2 * kKvKeysPerWg * p.d / 1024, chain_split_blocks(p, share), p.B * p.H);
    const int n_wg = chain_wgs(p, share);
    if (out_dt == CONVATTN_BF16)
        chain_reduce_kernel<bf16_t><<<grid, 256, 0, s>>>(p, share, n_wg, part, (bf16_t *)dk, (bf16_t *)dv);
    else
        chain_reduce_kernel<float><<<grid, 256, 0, s>>>(p, share, n_wg, part, (float *)dk, (float *)dv);
    return hipGetLastError();
}

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

hipError_t decode_combine(const Problem &p, int out_dt, const float *o_part, const float *m_part,
                          const float *l_part, void *o, float *m, float *l, hipStream_t s) {
    // Up to 16 splits are all in flight in one thread per column; more (few pairs over a long cache have hundreds) are taken by a
    // workgroup's threads together.  (Step of B1 H8 d64, us, walked before / in flight / together: N2048 in 8 splits 11.9 / 9.4 / -,
    // in 16 - / 9.7 / 9.9, in 32 - / 11.1 / 10.7.)
    const unsigned few = (unsigned)(p.B * p.H);
    if (p.n_splits <= 8) {
        if (out_dt == CONVATTN_BF16) combine_few_kernel<8, bf16_t><<<few, 128, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (bf16_t *)o, m, l);
        else combine_few_kernel<8, float><<<few, 128, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (float *)o, m, l);
        return hipGetLastError();
    }
    if (p.n_splits <= 16) {
        if (out_dt == CONVATTN_BF16) combine_few_kernel<16, bf16_t><<<few, 128, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (bf16_t *)o, m, l);
        else combine_few_kernel<16, float><<<few, 128, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (float *)o, m, l);
        return hipGetLastError();
    }
    const dim3 grid((unsigned)(p.B * p.H), (unsigned)((p.d + 31) / 32));
    if (out_dt == CONVATTN_BF16)
        combine_kernel<bf16_t><<<grid, 256, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (bf16_t *)o, m, l);
    else
        combine_kernel<float><<<grid, 256, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (float *)o, m, l);
    return hipGetLastError();
}

}  // namespace convattn
