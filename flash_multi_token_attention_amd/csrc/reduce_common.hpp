// Row statistics and reductions of the backward passes, for the kernels of their own and those that take them on the way.
#pragma once
#include "mfma_common.hpp"

namespace convattn {

// D = <dO, O>, LSE = M + log L.  16 lanes per query row, 8 elements (16 or 32 bytes) per lane:
// a wave reads 4 rows at a time with full-width loads; d is a multiple of 8 and at most 128.
template <typename T>
__device__ __forceinline__ void load8(const T *__restrict__ ptr, float (&v)[8]) {
    if constexpr (sizeof(T) == 2) {
        const uint4 raw = *reinterpret_cast<const uint4 *>(ptr);
        const unsigned int w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = __uint_as_float(w[i] << 16);
            v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    } else {
        const float4 a = *reinterpret_cast<const float4 *>(ptr);
        const float4 b = *reinterpret_cast<const float4 *>(ptr + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
}

// (block: of 256 threads and 16 rows)
template <typename TI, typename TO>
__device__ __forceinline__ void row_stats(size_t block, size_t rows, int d, const TO *__restrict__ O, const TI *__restrict__ dO,
                                          const float *__restrict__ M, const float *__restrict__ L, float *__restrict__ D,
                                          float *__restrict__ LSE) {
    const size_t row = block * 16 + (threadIdx.x >> 4);
    const int sub = threadIdx.x & 15;
    float s = 0.f;
    if (row < rows && sub * 8 < d) {
        float o[8], g[8];
        load8(O + row * d + sub * 8, o);
        load8(dO + row * d + sub * 8, g);
#pragma unroll
        for (int i = 0; i < 8; ++i) s = fmaf(o[i], g[i], s);
    }
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) s += __shfl_xor(s, m, 16);
    if (row < rows && sub == 0) {
        D[row] = s;
        LSE[row] = M[row] + __logf(L[row]);
    }
}

// dW[h][tap] = sum over (batch, tile) of the partials, in a fixed order: a workgroup takes 64 taps (block ty) of one head
// (lane = tap, so a partial is read with contiguous loads); chain w of the 16 that its waves share out adds the partials
// w, w + 16, ... in four independent sums, and the chains' sums are added in order.
constexpr int kDwChains = 16;
template <int THREADS>
__device__ __forceinline__ void dw_reduce_block(int B, int H, int n_tiles, int ntap, const float *__restrict__ part,
                                                float *__restrict__ dW, int h, int ty, float (*red)[64]) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tap = ty * 64 + lane;
    const int n = B * n_tiles;
    for (int w = wave; w < kDwChains; w += THREADS / 64) {
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        if (tap < ntap) {
            auto at = [&](int q) {
                const int b = q / n_tiles, t = q - b * n_tiles;
                return part[(((size_t)b * H + h) * n_tiles + t) * ntap + tap];
            };
            int q = w;
            for (; q + 3 * kDwChains < n; q += 4 * kDwChains) {
#pragma unroll
                for (int c = 0; c < 4; ++c) s[c] += at(q + kDwChains * c);
            }
            for (int c = 0; q < n; q += kDwChains, ++c) s[c] += at(q);
        }
        red[w][lane] = (s[0] + s[1]) + (s[2] + s[3]);
    }
    __syncthreads();
    if (wave == 0 && tap < ntap) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kDwChains; ++w) v += red[w][lane];
        dW[(size_t)h * ntap + tap] = v;
    }
}

// dK and dV of a key block whose row tiles several workgroups share: the partials added in the order of the rows.
// bx = 256 groups of 4 values of the block's dK, then dV.
template <typename TO>
__device__ __forceinline__ void chain_reduce_block(const Problem &p, int share, int n_wg, const float *__restrict__ part,
                                                   TO *__restrict__ dK, TO *__restrict__ dV, int bx, int kb, size_t bh) {
    const int parts = chain_parts(p, kb, share);
    if (parts == 1) return;
    int z = 0;
    for (int i = 0; i < kb; ++i) z += chain_parts(p, i, share);
    const int e = (bx * 256 + threadIdx.x) * 4, per = kKvKeysPerWg * p.d;   // (2 per is a multiple of 1024)
    const int is_v = e >= per, local = e - is_v * per, key = kb * kKvKeysPerWg + local / p.d - (is_v ? 8 : 0);
    if (key < 0 || key >= p.Nk) return;
    const float *src = part + (bh * n_wg + z) * 2 * per + e;
    float4 sum = *reinterpret_cast<const float4 *>(src);
    for (int i = 1; i < parts; ++i) {
        const float4 v = *reinterpret_cast<const float4 *>(src + (size_t)i * 2 * per);
        sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    TO *dst = (is_v ? dV : dK) + (bh * p.Nk + key) * p.d + local % p.d;
    if constexpr (sizeof(TO) == 2) {
        bf16x4 o = {(bf16_t)sum.x, (bf16_t)sum.y, (bf16_t)sum.z, (bf16_t)sum.w};
        *reinterpret_cast<bf16x4 *>(dst) = o;
    } else {
        *reinterpret_cast<float4 *>(dst) = sum;
    }
}

}  // namespace convattn
