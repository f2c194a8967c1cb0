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

// Merge of a few decode splits: one workgroup per (batch, head), one thread per output column walks the splits.
template <typename TO>
__global__ void combine_few_kernel(int n_splits, int d, const float *__restrict__ O_part,
                                   const float *__restrict__ M_part, const float *__restrict__ L_part,
                                   TO *__restrict__ O, float *__restrict__ M, float *__restrict__ L) {
    const size_t bh = blockIdx.x;
    const float *mp = M_part + bh * n_splits;
    const float *lp = L_part + bh * n_splits;
    float m = kNegInf;
    for (int s = 0; s < n_splits; ++s) m = fmaxf(m, mp[s]);
    float l = 0.f;
    for (int s = 0; s < n_splits; ++s) l += (mp[s] == kNegInf) ? 0.f : lp[s] * __expf(mp[s] - m);
    for (int c = threadIdx.x; c < d; c += blockDim.x) {
        float o = 0.f;
        for (int s = 0; s < n_splits; ++s)
            if (mp[s] != kNegInf) o = fmaf(O_part[(bh * n_splits + s) * d + c], __expf(mp[s] - m), o);
        O[bh * d + c] = from_f32<TO>(o / l);
    }
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

// Row tiles per workgroup of the split backward, or 0: one workgroup per key block.  In units of a row tile a workgroup
// costs its tiles, about 4.5 for set-up and wind-down and one more where its range ends inside the key block; the launch
// the longest workgroup or the CUs' even part of everything plus a third of the longest; the reduction kernel 6 to 8.
// (B2 H8 N1531 d64 11x11: 167 -> 109 us, B1 H8 N2048 d64 7x7: 169 -> 72, B1 H8 N1000 d128 6x11: 78 -> 32.)
// Sequences of less than 20 row tiles gain less than the reduction and its launch cost.  From 8192 rows on nothing is split, whatever
// the number of heads is: a head's results do not depend on how many others there are.
int chain_share(const Problem &p) {
    const int n_rt = chain_row_tiles(p), n_kb = mfma_kv_tiles(p);
    if (n_rt < 20 || p.Nq >= 8192 || p.B * (long long)p.H > 64) return 0;
    float none = 0.f, best = 0.f;
    int share = 0;
    for (int cut = 1; cut <= 8; cut += cut < 4 ? 1 : 2) {
        const int s = cut == 1 ? 0 : (n_rt + cut - 1) / cut;
        if (cut > 1 && s < 6) break;
        float total = 0.f, longest = 0.f;
        int jobs = 0;
        for (int kb = 0; kb < n_kb; ++kb) {
            const int len = chain_len(p, kb) > 0 ? chain_len(p, kb) : 0, parts = chain_parts(p, kb, s);
            const float one = (float)((len + parts - 1) / parts) + 4.5f + (parts > 1 ? 1.f : 0.f);
            longest = one > longest ? one : longest;
            total += one * parts;
            jobs += parts;
        }
        const float n = (float)p.B * p.H, even = total * n / 256.f + longest / 3.f;
        const float t = jobs * n <= 256.f || longest > even ? longest : even;
        if (cut == 1) none = best = t;
        else if (1.05f * t + 7.f < none && t < best) { best = t; share = s; }
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

hipError_t decode_combine(const Problem &p, int out_dt, const float *o_part, const float *m_part,
                          const float *l_part, void *o, float *m, float *l, hipStream_t s) {
    // (a serving step with many (batch, head) pairs has a handful of splits: the walk over them is shorter than
    // the second kernel's two reductions; few pairs over a long cache have hundreds)
    if (p.n_splits <= 8) {
        const unsigned few = (unsigned)(p.B * p.H);
        if (out_dt == CONVATTN_BF16)
            combine_few_kernel<bf16_t><<<few, 128, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (bf16_t *)o, m, l);
        else
            combine_few_kernel<float><<<few, 128, 0, s>>>(p.n_splits, p.d, o_part, m_part, l_part, (float *)o, m, l);
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
