// Row statistics of a backward pass, shared by the kernels that take them on the way.
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

}  // namespace convattn
