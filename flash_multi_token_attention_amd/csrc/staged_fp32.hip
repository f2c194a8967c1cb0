// fp32-arithmetic conv-attention with the score-sized matrices in global memory (gfx950): every supported shape, both
// input types, forward and whole backward.
//
// The kernels of generic_kernels.hip keep a tile's scores, convolution and probabilities in LDS and recompute them in
// each of three passes; their convolutions read one LDS word per two multiply-adds and a workgroup owns 16 rows
// (B1 H8 N1024 d64 6x11: 0.15 + 0.84 + 0.62 ms for about 0.06 ms of arithmetic).  Here every (row, key) pair is convolved once per
// pass, by workgroups of 64 rows x 64 keys that are independent of each other, so that short sequences fill the chip:
//   forward    window_kernel<fwd>: S = scale Q K^T with its halo (fp32 MFMA), C = window(S) -> C, row maxima of the tile
//              product_kernel<0>:  O = exp(C - M) V / L
//   backward   window_kernel<bwd>: S, C, P = exp(C - LSE), dP = dO V^T, dC = P (dP - D) -> P, dC; dW partial of the tile
//              unwindow_kernel:    dS = transposed window(dC)
//              product_kernel<1..3>: dQ = dS K, dV = P^T dO, dK = dS^T Q
// All operands, scores and sums are fp32, dW is summed in a fixed order, nothing is added with atomics.  The matrices take
// 4 bytes per pair (forward one, backward three of them; the whole square under the causal mask too).  Above the caller's
// workspace limit the Python ops run them by groups of heads; the other kernels run where one head does not fit.
#include "reduce_common.hpp"

namespace convattn {
namespace {

constexpr int NT = 256, TT = 64;                 // threads; rows and keys of a tile
constexpr int KC = 64;                           // columns of Q and K that a tile stages at a time: four workgroups per CU at d = 128 too
                                                 // (whole rows, two: B1 H8 N1024 d128 6x11 backward 99 -> 83 us, forward 60 -> 49)

struct StArgs {
    Problem p;
    int ld;              // row stride of the matrices (floats): Nk rounded up to whole tiles
    int n_rt, n_ct;      // tiles of 64 rows / keys
    float *c, *pm, *ds;  // C or dC; P; dS
    float *mx;           // forward: row maxima per tile column [BH][n_ct][Nq]
};

__device__ __forceinline__ f32x4 load4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }
__device__ __forceinline__ f32x4 load4(const bf16_t *p) {
    const bf16x4 v = *reinterpret_cast<const bf16x4 *>(p);
    return (f32x4){(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}
__host__ __device__ inline int round16(int d) { return (d + 15) & ~15; }

// dst[r][0 .. width) = columns col0 .. of row row0 + r of src for r < rows; zeros outside [0, N) and past d
template <typename TI>
__device__ __forceinline__ void stage_rows(float *dst, int st, const TI *__restrict__ src, int row0, int rows, int N, int d, int col0, int width) {
    const int q = width / 4;
    constexpr int U = 8;   // loads in flight per thread
    if (NT % q == 0) {
        const int c = (threadIdx.x % q) * 4, step = NT / q;
        for (int r = threadIdx.x / q; r < rows; r += U * step) {
            f32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int g = row0 + r + u * step;
                v[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
                if (r + u * step < rows && g >= 0 && g < N && col0 + c < d) v[u] = load4(src + (size_t)g * d + col0 + c);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (r + u * step < rows) *reinterpret_cast<f32x4 *>(dst + (r + u * step) * st + c) = v[u];
        }
        return;
    }
    for (int i = threadIdx.x; i < rows * q; i += NT) {
        const int r = i / q, c = (i - r * q) * 4, g = row0 + r;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (g >= 0 && g < N && col0 + c < d) v = load4(src + (size_t)g * d + col0 + c);
        *reinterpret_cast<f32x4 *>(dst + r * st + c) = v;
    }
}

// acc (lane (g, n): rows 4g .. 4g+3 of A, row n of B_u) = A B_u^T over k < K (a multiple of 16), both with k along
// their rows in LDS.  A lane reads four consecutive k of a row (k slot g of MFMA s = element 4g + s of the sixteen); row strides
// are 4 mod 64 floats for d = 64, 128: sixteen rows on sixteen bank quads.
template <int NB>
__device__ __forceinline__ void mma_nt(f32x4 (&acc)[NB], const float *a, const float *const (&b)[NB], int K) {
    for (int k = 0; k < K; k += 16) {
        const f32x4 av = *reinterpret_cast<const f32x4 *>(a + k);
        f32x4 bv[NB];
#pragma unroll
        for (int u = 0; u < NB; ++u) bv[u] = *reinterpret_cast<const f32x4 *>(b[u] + k);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int u = 0; u < NB; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], bv[u][s], acc[u], 0, 0, 0);
    }
}

// The head's window in LDS, rows of round4(c_k) floats (zeros behind the taps); FLIP: turned by 180 degrees
__host__ __device__ inline int win_stride(int c_k) { return (c_k + 3) & ~3; }
template <bool FLIP>
__device__ __forceinline__ void stage_window(float *ws, const float *__restrict__ w, int c_q, int c_k) {
    const int wst = win_stride(c_k);
    for (int i = threadIdx.x; i < c_q * wst; i += NT) {
        const int a = i / wst, b = i - a * wst;
        ws[i] = b < c_k ? w[(FLIP ? c_q - 1 - a : a) * c_k + (FLIP ? c_k - 1 - b : b)] : 0.f;
    }
}

// out[o][k] = sum_ab w(a, b) x[(o + a) * st + k + b] for a 4 x 4 patch of outputs (x and w in LDS, 16-byte aligned).  A ring of
// four rows in registers: one new row and one row of weights (16-byte reads, the weights a broadcast) per 16 CK multiply-adds;
// weights by scalar loads made every row wait for one.  CK = 0: any width, one column at a time.
// Each tap row is summed by itself: one chain over the window (121 terms for 11 x 11) raised the errors of dQ and dK against 64
// bits by 4 to 12 % (B1 H4 N700 d128 11 x 11 dQ 5.03 -> 5.66e-7 of its norm, B1 H8 N64 d64 6 x 11 3.43 -> 3.79e-7).  It costs one
// addition to CK multiply-adds (training step of B1 H8 N1024 d64 6 x 11 160.7 -> 162.5 us), and the row sums of one output row at a
// time, or unwindow_kernel's registers do not hold them.
template <int CK>
__device__ __forceinline__ void patch_conv(float (&out)[4][4], const float *w, int c_q, int c_k, const float *x, int st) {
#pragma unroll
    for (int o = 0; o < 4; ++o)
#pragma unroll
        for (int k = 0; k < 4; ++k) out[o][k] = 0.f;
    if constexpr (CK > 0) {
        constexpr int RW = (CK + 3 + 3) / 4, WQ = (CK + 3) / 4;
        f32x4 ring[4][RW];
        auto load = [&](int slot, int r) {
#pragma unroll
            for (int i = 0; i < RW; ++i) ring[slot][i] = *reinterpret_cast<const f32x4 *>(x + r * st + 4 * i);
        };
#pragma unroll
        for (int r = 0; r < 3; ++r) load(r, r);
        for (int a0 = 0; a0 < c_q; a0 += 4) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                if (a0 + s < c_q) {
                    f32x4 wv[WQ];
#pragma unroll
                    for (int i = 0; i < WQ; ++i) wv[i] = *reinterpret_cast<const f32x4 *>(w + (a0 + s) * (4 * WQ) + 4 * i);
                    load((s + 3) & 3, a0 + s + 3);
#pragma unroll
                    for (int o = 0; o < 4; ++o) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            float r = wv[0][0] * ring[(s + o) & 3][k / 4][k & 3];
#pragma unroll
                            for (int b = 1; b < CK; ++b) r = fmaf(wv[b / 4][b & 3], ring[(s + o) & 3][(k + b) / 4][(k + b) & 3], r);
                            out[o][k] += r;
                        }
                    }
                }
            }
        }
    } else {
        const int wst = win_stride(c_k);
        for (int a = 0; a < c_q; ++a)
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                float row[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (int b = 0; b < c_k; ++b)
#pragma unroll
                    for (int k = 0; k < 4; ++k) row[k] = fmaf(w[a * wst + b], x[(o + a) * st + k + b], row[k]);
#pragma unroll
                for (int k = 0; k < 4; ++k) out[o][k] += row[k];
            }
    }
}
__device__ __forceinline__ void patch_conv_any(float (&out)[4][4], const float *w, int c_q, int c_k, const float *x, int st) {
    switch (c_k) {   // (workgroup-uniform)
        case 1: patch_conv<1>(out, w, c_q, c_k, x, st); break;
        case 3: patch_conv<3>(out, w, c_q, c_k, x, st); break;
        case 5: patch_conv<5>(out, w, c_q, c_k, x, st); break;
        case 7: patch_conv<7>(out, w, c_q, c_k, x, st); break;
        case 9: patch_conv<9>(out, w, c_q, c_k, x, st); break;
        case 11: patch_conv<11>(out, w, c_q, c_k, x, st); break;
        case 13: patch_conv<13>(out, w, c_q, c_k, x, st); break;
        case 15: patch_conv<15>(out, w, c_q, c_k, x, st); break;
        default: patch_conv<0>(out, w, c_q, c_k, x, st); break;
    }
}

// Tile `id` of a launch of BH * tiles workgroups: every workgroup has work (a square grid under the causal mask would leave
// half of them empty, and unevenly over the XCDs, which take workgroups in turn); row tiles from the last on.
__host__ __device__ inline long long tile_count(bool causal, int n_rt, int n_ct) { return causal ? (long long)n_rt * (n_rt + 1) / 2 : (long long)n_rt * n_ct; }
__device__ __forceinline__ void find_tile(const Problem &p, int n_rt, int n_ct, size_t &bh, int &rt, int &ct, long long &tile) {
    const long long tiles = tile_count(p.causal != 0, n_rt, n_ct);
    bh = blockIdx.x / tiles;
    tile = tiles - 1 - (long long)(blockIdx.x - bh * tiles);
    if (p.causal) {
        int r = (int)((sqrtf(8.f * (float)tile + 1.f) - 1.f) * 0.5f);
        while ((long long)(r + 1) * (r + 2) / 2 <= tile) ++r;
        while ((long long)r * (r + 1) / 2 > tile) --r;
        rt = r;
        ct = (int)(tile - (long long)r * (r + 1) / 2);
    } else {
        rt = (int)(tile / n_ct);
        ct = (int)(tile - (long long)rt * n_ct);
    }
    rt = __builtin_amdgcn_readfirstlane(rt);
    ct = __builtin_amdgcn_readfirstlane(ct);
}

template <int ROR> __device__ __forceinline__ float row16_rot(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + ROR, 0xf, 0xf, true));
}
// dW of one tile.  A unit of work is a tap row over half of the tile's rows; a wave takes the units wave, wave + 4, ..., a lane
// four columns of eight rows: acc[b] = sum over them of dC[i][j] S[i + a][j + b].  The sixteen lanes of a row are added by
// rotations (vector-ALU speed; a shuffle per step would pass the LDS), the eight sums of a tap in order at the end.
template <int CK>
__device__ __forceinline__ void tile_dw(float *__restrict__ part, float *red, int c_q, int c_k, const float *dc, int dst, const float *S, int sst) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, tx = lane & 15, ty = lane >> 4;
    if constexpr (CK > 0) {
        constexpr int RW = (CK + 3 + 3) / 4;
        for (int u = wave; u < 2 * c_q; u += NT / 64) {
            const int a = u >> 1, i0 = (u & 1) * (TT / 2) + ty * 8;
            float acc[CK];
#pragma unroll
            for (int b = 0; b < CK; ++b) acc[b] = 0.f;
#pragma unroll 2
            for (int i = i0; i < i0 + 8; ++i) {
                const f32x4 d = *reinterpret_cast<const f32x4 *>(dc + i * dst + 4 * tx);
                f32x4 s[RW];
#pragma unroll
                for (int q = 0; q < RW; ++q) s[q] = *reinterpret_cast<const f32x4 *>(S + (i + a) * sst + 4 * tx + 4 * q);
#pragma unroll
                for (int b = 0; b < CK; ++b)
#pragma unroll
                    for (int k = 0; k < 4; ++k) acc[b] = fmaf(d[k], s[(k + b) / 4][(k + b) & 3], acc[b]);
            }
#pragma unroll
            for (int b = 0; b < CK; ++b) {
                float v = acc[b];
                v += row16_rot<8>(v);
                v += row16_rot<4>(v);
                v += row16_rot<2>(v);
                v += row16_rot<1>(v);
                if (tx == 0) red[(a * CK + b) * 8 + (u & 1) * 4 + ty] = v;
            }
        }
        __syncthreads();
        for (int tap = threadIdx.x; tap < c_q * CK; tap += NT) {
            float v = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) v += red[tap * 8 + e];
            part[tap] = v;
        }
    } else {   // any width: a wave per tap
        for (int tap = wave; tap < c_q * c_k; tap += NT / 64) {
            const int a = tap / c_k, b = tap - a * c_k;
            float s = 0.f;
            for (int i = 0; i < TT; ++i) s = fmaf(dc[i * dst + lane], S[(i + a) * sst + lane + b], s);
            s = wave_sum(s);
            if (lane == 0) part[tap] = s;
        }
    }
}
__device__ __forceinline__ void tile_dw_any(float *__restrict__ part, float *red, int c_q, int c_k, const float *dc, int dst, const float *S,
                                            int sst) {
    switch (c_k) {   // (workgroup-uniform)
        case 1: tile_dw<1>(part, red, c_q, c_k, dc, dst, S, sst); break;
        case 3: tile_dw<3>(part, red, c_q, c_k, dc, dst, S, sst); break;
        case 5: tile_dw<5>(part, red, c_q, c_k, dc, dst, S, sst); break;
        case 7: tile_dw<7>(part, red, c_q, c_k, dc, dst, S, sst); break;
        case 9: tile_dw<9>(part, red, c_q, c_k, dc, dst, S, sst); break;
        case 11: tile_dw<11>(part, red, c_q, c_k, dc, dst, S, sst); break;
        case 13: tile_dw<13>(part, red, c_q, c_k, dc, dst, S, sst); break;
        case 15: tile_dw<15>(part, red, c_q, c_k, dc, dst, S, sst); break;
        default: tile_dw<0>(part, red, c_q, c_k, dc, dst, S, sst); break;
    }
}

// LDS of window_kernel: KC columns of the rows of Q and K, then in their place dP / dC (backward), the sums of dW and the score tile with its halo.
// (The score tile beside the rows, and rows of dO and V staged as well, took 60 KB at d = 64: two workgroups per CU, and one at
// d = 128.  Now 39: B1 H8 N1024 d64 6x11 backward 73 -> 58 us, forward 42 -> 36.)
struct WinLds {
    int dst, sst, k_f, dp_f, w_f, s_f, total_f;   // floats
};
__host__ __device__ inline WinLds win_lds(const Problem &p, bool bwd) {
    WinLds l;
    l.dst = (round16(p.d) < KC ? round16(p.d) : KC) + 4;
    // a patch reads whole 16-byte quantities: columns 60 .. 60 + c_k + 3 rounded up
    l.sst = TT - 4 + ((p.c_k + 3 + 3) & ~3);
    l.w_f = 0;                                            // window
    const int rows = p.c_q * win_stride(p.c_k);           // first float of the rows of Q
    l.k_f = rows + (TT + p.pq) * l.dst;
    l.s_f = rows;                                         // score tile
    l.dp_f = l.s_f + (TT + p.pq) * l.sst;
    const int one = l.k_f + (TT + 2 * p.pk) * l.dst;
    const int two = l.dp_f + (bwd ? TT * (TT + 4) + (p.c_k <= 15 ? 8 * p.c_q * p.c_k : 0) : 0);
    l.total_f = one > two ? one : two;
    return l;
}

// One tile of 64 rows x 64 keys: S with the window's halo, C = window(S).
//   BWD = false: C (-inf where masked) and the rows' maxima of the tile
//   BWD = true:  P, dC and the tile's dW
// Held to four workgroups per CU, as many as the LDS has room for at d = 64 (141 registers fall to 125, none spilled): B1 H2 N1294
// d64 6x11 not causal 150 -> 143 us, shapes whose workgroups are fewer or whose rows are longer the same.
template <bool BWD, typename TI>
__global__ __launch_bounds__(NT, 4) void window_kernel(StArgs a, const TI *__restrict__ Q, const TI *__restrict__ K, const TI *__restrict__ V,
                                                    const TI *__restrict__ dO, const float *__restrict__ D, const float *__restrict__ LSE,
                                                    const float *__restrict__ W, float *__restrict__ dw_part) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const Problem &p = a.p;
    size_t bh;
    int rt, ct;
    long long tile;
    find_tile(p, a.n_rt, a.n_ct, bh, rt, ct, tile);
    const int h = (int)(bh % p.H), r0 = rt * TT, c0 = ct * TT, d = p.d, pq = p.pq, pk = p.pk, Kd = round16(d);
    const WinLds L = win_lds(p, BWD);
    float *Qs = lds + L.s_f, *Ks = lds + L.k_f, *Ss = lds + L.s_f, *Ws = lds + L.w_f, *dPs = lds + L.dp_f;   // dP: [64][68]
    constexpr int PST = TT + 4;
    const int nr = TT + pq, nc = TT + 2 * pk;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, n = lane & 15;

    stage_window<false>(Ws, W + (size_t)h * p.c_q * p.c_k, p.c_q, p.c_k);
    // score blocks of 16 rows x 32 keys, held until the rows have been read by everyone
    constexpr int HELD = 4;   // (at most 5 x 3 blocks for four waves)
    const int nrb = (nr + 15) / 16, ncb = (nc + 15) / 16, ncp = (ncb + 1) / 2;
    f32x4 sc[HELD][2];
#pragma unroll
    for (int x = 0; x < HELD; ++x) sc[x][0] = sc[x][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < Kd; k0 += KC) {
        const int width = min(KC, Kd - k0);
        if (k0) __syncthreads();
        stage_rows(Qs, L.dst, Q + bh * p.Nq * d, r0 - pq, nr, p.Nq, d, k0, width);
        stage_rows(Ks, L.dst, K + bh * p.Nk * d, c0 - pk, nc, p.Nk, d, k0, width);
        __syncthreads();
#pragma unroll
        for (int x = 0; x < HELD; ++x) {
            const int it = wave + x * (NT / 64);
            if (it < nrb * ncp) {
                const int rb = it / ncp, cb = (it - rb * ncp) * 2;
                const float *bp[2] = {Ks + min(cb * 16 + n, nc - 1) * L.dst + 4 * g, Ks + min(cb * 16 + 16 + n, nc - 1) * L.dst + 4 * g};
                mma_nt<2>(sc[x], Qs + min(rb * 16 + n, nr - 1) * L.dst + 4 * g, bp, width);
            }
        }
    }
    f32x4 dp_acc[4];
    if constexpr (BWD) {
        // dP = dO V^T, the operands as they lie in memory (sixteen consecutive k of sixteen rows per load)
        const TI *gp = dO + (bh * p.Nq + min(r0 + wave * 16 + n, p.Nq - 1)) * d, *vp[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            dp_acc[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
            vp[u] = V + (bh * p.Nk + min(c0 + u * 16 + n, p.Nk - 1)) * d;   // (pairs past the last row or key are dropped below)
        }
        f32x4 av, bv[4];
        auto fetch = [&](int k) {
            const bool in = k + 4 * g < d;
            const int at = in ? k + 4 * g : 0;
            av = load4(gp + at);
            if (!in) av = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 4; ++u) bv[u] = load4(vp[u] + at);
        };
        fetch(0);
        for (int k = 0; k < Kd; k += 16) {
            const f32x4 a0 = av, b0[4] = {bv[0], bv[1], bv[2], bv[3]};
            fetch(min(k + 16, Kd - 16));
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int u = 0; u < 4; ++u) dp_acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[s], b0[u][s], dp_acc[u], 0, 0, 0);
        }
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < HELD; ++x) {
        const int it = wave + x * (NT / 64);
        if (it < nrb * ncp) {
            const int rb = it / ncp, cb = (it - rb * ncp) * 2;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = rb * 16 + 4 * g + r, j = (cb + u) * 16 + n;
                    if (i < nr && j < nc) Ss[i * L.sst + j] = p.causal && c0 - pk + j > r0 - pq + i ? 0.f : sc[x][u][r] * p.scale;
                }
        }
    }
    // (columns past the halo that a patch's last 16 bytes touch: multiplied by nothing, but not to be NaN patterns either)
    for (int r = tid; r < nr; r += NT)
        for (int c = nc; c < L.sst; ++c) Ss[r * L.sst + c] = 0.f;
    if constexpr (BWD) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) dPs[(wave * 16 + 4 * g + r) * PST + u * 16 + n] = dp_acc[u][r];
    }
    __syncthreads();
    // ---- window: a thread has rows 4 ty .., keys 4 tx .. ----
    const int tx = tid & 15, ty = tid >> 4, key0 = c0 + 4 * tx;
    float c[4][4];
    patch_conv_any(c, Ws, p.c_q, p.c_k, Ss + 4 * ty * L.sst + 4 * tx, L.sst);
#pragma unroll
    for (int o = 0; o < 4; ++o) {
        const int row = r0 + 4 * ty + o;
        const size_t at = (bh * p.Nq + row) * a.ld + key0;
        if constexpr (!BWD) {
            f32x4 v;
            float m = kNegInf;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[k] = key0 + k >= p.Nk || (p.causal && key0 + k > row) ? kNegInf : c[o][k];
                m = fmaxf(m, v[k]);
            }
#pragma unroll
            for (int s = 8; s > 0; s >>= 1) m = fmaxf(m, __shfl_xor(m, s, 16));
            if (row < p.Nq) {
                *reinterpret_cast<f32x4 *>(a.c + at) = v;
                if (tx == 0) a.mx[(bh * a.n_ct + ct) * p.Nq + row] = m;
            }
        } else {
            const bool ok = row < p.Nq;
            const float lse = ok ? LSE[bh * p.Nq + row] : 0.f, dd = ok ? D[bh * p.Nq + row] : 0.f;
            float *dp = dPs + (4 * ty + o) * PST + 4 * tx;
            f32x4 v = *reinterpret_cast<const f32x4 *>(dp), pv;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                pv[k] = !ok || key0 + k >= p.Nk || (p.causal && key0 + k > row) ? 0.f : __expf(c[o][k] - lse);
                v[k] = pv[k] * (v[k] - dd);
            }
            *reinterpret_cast<f32x4 *>(dp) = v;
            if (ok) {
                *reinterpret_cast<f32x4 *>(a.pm + at) = pv;
                *reinterpret_cast<f32x4 *>(a.c + at) = v;
            }
        }
    }
    if (BWD && dw_part) {
        __syncthreads();
        tile_dw_any(dw_part + (bh * tile_count(p.causal != 0, a.n_rt, a.n_ct) + tile) * p.c_q * p.c_k, dPs + TT * PST, p.c_q, p.c_k, dPs, PST, Ss, L.sst);
    }
}

// dS[r][c] = sum_ab W[a][b] dC[r - a + pq][c - b + pk]: the window turned by 180 degrees over the rows from r on and the keys from
// c - pk on.  A workgroup waits for its tile's rows first and multiplies afterwards, so what covers the wait is the others on the
// CU: held to five (96 registers, 160 values spilled around the taps), B1 H8 N1024 d64's 1088 workgroups are all resident at once
// (23 -> 19 us at four; B1 H2 N2002 d128 21 -> 17; with a sum for each tap row the whole step takes 162.5 us, at four 165.6).
__global__ __launch_bounds__(NT, 5) void unwindow_kernel(StArgs a, const float *__restrict__ W) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const Problem &p = a.p;
    size_t bh;
    int rt, ct;
    long long tile;
    find_tile(p, a.n_rt, a.n_ct, bh, rt, ct, tile);
    const int h = (int)(bh % p.H), r0 = rt * TT, c0 = ct * TT, sst = win_lds(p, true).sst, nr = TT + p.pq, tid = threadIdx.x;
    float *Ws = lds + nr * sst;
    stage_window<true>(Ws, W + (size_t)h * p.c_q * p.c_k, p.c_q, p.c_k);
    {
        // a wave per row, two columns per lane (a row is at most 96 wide), six rows in flight
        constexpr int U = 6;
        const int wave = tid >> 6, lane = tid & 63;
        for (int r = wave; r < nr; r += U * (NT / 64)) {
            float v[U][2];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int row = r0 + r + u * (NT / 64), x = lane + 64 * e, key = c0 - p.pk + x;
                    // (pairs after the row's position were not written: their dC is zero)
                    const bool ok = r + u * (NT / 64) < nr && x < sst && row < p.Nq && key >= 0 && key < p.Nk && !(p.causal && key > row);
                    v[u][e] = ok ? a.c[(bh * p.Nq + row) * a.ld + key] : 0.f;
                }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    if (r + u * (NT / 64) < nr && lane + 64 * e < sst) lds[(r + u * (NT / 64)) * sst + lane + 64 * e] = v[u][e];
        }
    }
    __syncthreads();
    const int tx = tid & 15, ty = tid >> 4, key0 = c0 + 4 * tx;
    float c[4][4];
    patch_conv_any(c, Ws, p.c_q, p.c_k, lds + 4 * ty * sst + 4 * tx, sst);
#pragma unroll
    for (int o = 0; o < 4; ++o) {
        const int row = r0 + 4 * ty + o;
        if (row < p.Nq) {
            f32x4 v;
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = key0 + k >= p.Nk || (p.causal && key0 + k > row) ? 0.f : c[o][k];
            *reinterpret_cast<f32x4 *>(a.ds + (bh * p.Nq + row) * a.ld + key0) = v;
        }
    }
}

// Products with a score-sized matrix X [rows][keys]: 32 rows (or keys) x d per workgroup of 8 waves, 64 of the contraction per
// step:
//   KIND 0: O = exp(C - M) V / L (also M, L)      1: dQ = scale dS K       (X as it lies)
//   KIND 2: dV = P^T dO                           3: dK = scale dS^T Q     (X turned)
// A wave has 16 rows of the result, all of d and one quarter of each step, the quarters are added at the end: a short sequence
// has few row tiles, and the longest walk is the launch (B1 H8 N1024 d64 forward: 64 rows and steps of 32 37 us, 32 rows and
// steps of 64 22 us).  The next step's operands are loaded into registers under this one's products.
// Steps of 64 instead of 128 leave room for more workgroups per CU (d = 64 three -> four, d = 128 one -> two): backward B1 H8 N2048 d64 98 -> 86 us,
// B1 H8 N1024 d128 64 -> 48 (both with the order of bwd_product_kernel), forward of the latter 32 -> 30.
constexpr int PM = 32, PKS = 64, PNT = 512;
template <int DBLK> struct ProdLds {
    static constexpr int BST = DBLK * 16 + 4, AST = PKS + 4, TST = PM + 4, hand_f = 3 * 2 * DBLK * 64 * 4;
    static constexpr int a_f = PM * AST > PKS * TST ? PM * AST : PKS * TST, total_f = a_f + (PKS * BST > hand_f ? PKS * BST : hand_f);
};
template <int KIND, int DBLK, typename TI, typename TO>
__device__ __forceinline__ void product(const StArgs &a, float *lds, size_t bh, int mt, const float *__restrict__ X, const TI *__restrict__ Y,
                                        TO *__restrict__ out, float *__restrict__ M, float *__restrict__ L) {
    using T = ProdLds<DBLK>;
    constexpr bool TURN = KIND >= 2;
    const Problem &p = a.p;
    const int d = p.d, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int mb = wave & 1, quarter = wave >> 1;
    const int m0 = mt * PM, NM = TURN ? p.Nk : p.Nq, NK = TURN ? p.Nq : p.Nk;
    // contraction range in whole steps: keys up to the rows' last, or rows from the tile of the keys' first
    const int k_begin = TURN && p.causal ? m0 / TT * TT : 0, k_end = !TURN && p.causal ? min(p.Nk, m0 + PM) : NK;
    const int x_end = p.causal ? (m0 / TT + 1) * TT : a.ld;   // (as it lies) columns that were written
    const float *Xb = X + bh * p.Nq * a.ld;
    const TI *Yb = Y + bh * NK * d;
    float *As = lds, *Bs = lds + T::a_f;

    // staging: A as it lies: row tid / 16, columns 4 (tid % 16) ..; turned: row tid / 8, columns 4 (tid % 8) ..
    const int ar = TURN ? tid >> 3 : tid >> 4, ac = TURN ? 4 * (tid & 7) : 4 * (tid & 15);
    constexpr int BQ = PKS * DBLK * 4 / PNT;          // 16-byte quantities of Y per thread
    float mrow = 0.f, lsum = 0.f;
    if constexpr (KIND == 0) {
        const int row = min(m0 + ar, p.Nq - 1);
        mrow = kNegInf;
        for (int t = tid & 15; t * TT < k_end; t += 16) mrow = fmaxf(mrow, a.mx[(bh * a.n_ct + t) * p.Nq + row]);
#pragma unroll
        for (int s = 8; s > 0; s >>= 1) mrow = fmaxf(mrow, __shfl_xor(mrow, s, 16));
    }
    f32x4 xa, yb[BQ];
    auto load = [&](int k0) {
        if constexpr (TURN) {
            const int row = k0 + ar;
            xa = (f32x4){0.f, 0.f, 0.f, 0.f};
            if (row < p.Nq) xa = *reinterpret_cast<const f32x4 *>(Xb + (size_t)row * a.ld + m0 + ac);
        } else {
            // (a step may end past the row's last written tile, or past the matrix: -inf and 0 there)
            const int key = k0 + ac;
            xa = KIND == 0 ? (f32x4){kNegInf, kNegInf, kNegInf, kNegInf} : (f32x4){0.f, 0.f, 0.f, 0.f};
            if (key < x_end) xa = *reinterpret_cast<const f32x4 *>(Xb + (size_t)min(m0 + ar, p.Nq - 1) * a.ld + key);
        }
#pragma unroll
        for (int i = 0; i < BQ; ++i) {
            const int q = tid + i * PNT, r = q / (DBLK * 4), c = (q - r * (DBLK * 4)) * 4;
            yb[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
            if (k0 + r < NK && c < d) yb[i] = load4(Yb + (size_t)(k0 + r) * d + c);
        }
    };
    f32x4 acc[DBLK];
#pragma unroll
    for (int u = 0; u < DBLK; ++u) acc[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
    load(k_begin);
    for (int k0 = k_begin; k0 < k_end; k0 += PKS) {
        if constexpr (KIND == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                xa[e] = __expf(xa[e] - mrow);
                lsum += xa[e];
            }
        }
        *reinterpret_cast<f32x4 *>(As + ar * (TURN ? T::TST : T::AST) + ac) = xa;
#pragma unroll
        for (int i = 0; i < BQ; ++i) {
            const int q = tid + i * PNT, r = q / (DBLK * 4), c = (q - r * (DBLK * 4)) * 4;
            *reinterpret_cast<f32x4 *>(Bs + r * T::BST + c) = yb[i];
        }
        __syncthreads();
        if (k0 + PKS < k_end) load(k0 + PKS);
#pragma unroll
        for (int kk = quarter * (PKS / 4); kk < quarter * (PKS / 4) + PKS / 4; kk += 16) {
            f32x4 av;
            if constexpr (TURN) {
#pragma unroll
                for (int s = 0; s < 4; ++s) av[s] = As[(kk + 4 * g + s) * T::TST + mb * 16 + n];
            } else {
                av = *reinterpret_cast<const f32x4 *>(As + (mb * 16 + n) * T::AST + kk + 4 * g);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int u = 0; u < DBLK; ++u)
                    acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], Bs[(kk + 4 * g + s) * T::BST + u * 16 + n], acc[u], 0, 0, 0);
        }
        __syncthreads();
    }
    // the other quarters to the first's waves; row sums
    f32x4 *hand = reinterpret_cast<f32x4 *>(Bs);
    if (quarter) {
#pragma unroll
        for (int u = 0; u < DBLK; ++u) hand[(((quarter - 1) * 2 + mb) * DBLK + u) * 64 + lane] = acc[u];
    }
    if constexpr (KIND == 0) {
#pragma unroll
        for (int s = 8; s > 0; s >>= 1) lsum += __shfl_xor(lsum, s, 16);
        if ((tid & 15) == 0) {
            As[ar] = lsum;
            if (m0 + ar < p.Nq) { M[bh * p.Nq + m0 + ar] = mrow; L[bh * p.Nq + m0 + ar] = lsum; }
        }
    }
    __syncthreads();
    if (quarter) return;
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int u = 0; u < DBLK; ++u) acc[u] += hand[((q * 2 + mb) * DBLK + u) * 64 + lane];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = mb * 16 + 4 * g + r;
        const float f = KIND == 0 ? 1.f / As[i] : KIND == 2 ? 1.f : p.scale;
        if (m0 + i < NM) {
#pragma unroll
            for (int u = 0; u < DBLK; ++u)
                if (u * 16 + n < d) out[(bh * NM + m0 + i) * d + u * 16 + n] = from_f32<TO>(acc[u][r] * f);
        }
    }
}

template <int DBLK, typename TI, typename TO>
__global__ __launch_bounds__(PNT) void fwd_product_kernel(StArgs a, const TI *__restrict__ V, TO *__restrict__ O, float *__restrict__ M,
                                                         float *__restrict__ L) {
    __shared__ __attribute__((aligned(16))) float lds[ProdLds<DBLK>::total_f];
    product<0, DBLK, TI, TO>(a, lds, blockIdx.x, gridDim.y - 1 - blockIdx.y, a.c, V, O, M, L);   // longest (causal) tiles first
}
// y = the products that are wanted, z = row or key tiles: the workgroups of all products come in the order of their length under
// the causal mask, the longest first (one product after the other B1 H8 N1024 d64 took 37 us, in this order 27).  The z behind the tiles
// sum dW's partials (x = head): a launch of their own took 5 us of the 162 of that shape's training step.  At d = 128 held to two workgroups
// per CU (126 registers instead of 138; 2 and 1 per CU: B1 H8 N2048 161 and 182 us, N1024 48 and 52, B1 H2 N2000, of 378 workgroups, 65 and 54).
template <int DBLK, typename TI, typename TO>
__global__ __launch_bounds__(PNT, 4) void bwd_product_kernel(StArgs a, const TI *__restrict__ Q, const TI *__restrict__ K, const TI *__restrict__ dO,
                                                         TO *__restrict__ dQ, TO *__restrict__ dK, TO *__restrict__ dV, int n_tiles,
                                                         const float *__restrict__ dw_part, float *__restrict__ dW) {
    __shared__ __attribute__((aligned(16))) float lds[ProdLds<DBLK>::total_f];
    static_assert(ProdLds<DBLK>::total_f >= kDwChains * 64, "room for the dW chains");
    const int t = blockIdx.z, which = blockIdx.y + (dQ ? 0 : 1), rows = (a.p.Nq + PM - 1) / PM, keys = (a.p.Nk + PM - 1) / PM;
    if (t >= max(rows, keys)) {
        const int ntap = a.p.c_q * a.p.c_k;
        if (blockIdx.y != 0 || (int)blockIdx.x >= a.p.H) return;
        for (int ty = t - max(rows, keys); ty * 64 < ntap; ty += gridDim.z - max(rows, keys)) {
            dw_reduce_block<PNT>(a.p.B, a.p.H, n_tiles, ntap, dw_part, dW, blockIdx.x, ty, reinterpret_cast<float (*)[64]>(lds));
            __syncthreads();
        }
    } else if (which == 0) {
        if (t < rows) product<1, DBLK, TI, TO>(a, lds, blockIdx.x, rows - 1 - t, a.ds, K, dQ, nullptr, nullptr);
    } else if (which == 1) {
        if (t < keys) product<2, DBLK, TI, TO>(a, lds, blockIdx.x, t, a.pm, dO, dV, nullptr, nullptr);
    } else {
        if (t < keys) product<3, DBLK, TI, TO>(a, lds, blockIdx.x, t, a.ds, Q, dK, nullptr, nullptr);
    }
}

StArgs make_args(const Problem &p) {
    StArgs a{};
    a.p = p;
    a.n_rt = (p.Nq + TT - 1) / TT;
    a.n_ct = (p.Nk + TT - 1) / TT;
    a.ld = a.n_ct * TT;
    return a;
}
size_t matrix_bytes(const StArgs &a) { return ((size_t)a.p.B * a.p.H * a.p.Nq * a.ld * sizeof(float) + 255) / 256 * 256; }
size_t dw_tiles(const StArgs &a) { return (size_t)tile_count(a.p.causal != 0, a.n_rt, a.n_ct); }

template <bool BWD, typename TI>
hipError_t launch_window(const StArgs &a, const void *q, const void *k, const void *v, const void *d_o, const float *D, const float *lse,
                         const float *w, float *part, hipStream_t s) {
    hipError_t e = set_max_lds_once<window_kernel<BWD, TI>>((int)kLdsBytes);
    if (e != hipSuccess) return e;
    window_kernel<BWD, TI><<<dim3((unsigned)((size_t)a.p.B * a.p.H * dw_tiles(a))), NT, win_lds(a.p, BWD).total_f * sizeof(float), s>>>(
        a, (const TI *)q, (const TI *)k, (const TI *)v, (const TI *)d_o, D, lse, w, part);
    return hipGetLastError();
}

}  // namespace

// Windows and sizes the staged kernels take: everything validate() lets through that fits their LDS and grids.
bool staged_ok(const Problem &p) {
    const StArgs a = make_args(p);
    const double pairs = (double)p.B * p.H, most = 4294967295.0;   // threads of a launch along x
    return (size_t)win_lds(p, true).total_f * sizeof(float) <= kLdsBytes && 2 * a.n_rt <= 65535 && 2 * a.n_ct <= 65535 &&
           pairs * (double)dw_tiles(a) * NT <= most && pairs * PNT <= most && (!p.causal || p.Nq == p.Nk);
}
size_t staged_fwd_bytes(const Problem &p) {
    const StArgs a = make_args(p);
    return matrix_bytes(a) + (size_t)p.B * p.H * a.n_ct * p.Nq * sizeof(float);
}
size_t staged_bwd_bytes(const Problem &p) {
    const StArgs a = make_args(p);
    return 3 * matrix_bytes(a) + (size_t)p.B * p.H * dw_tiles(a) * p.c_q * p.c_k * sizeof(float);
}

#define STAGED_IO(CALL)                                                                       \
    (in_dt == CONVATTN_BF16 ? (out_dt == CONVATTN_BF16 ? CALL(bf16_t, bf16_t) : CALL(bf16_t, float)) \
                            : (out_dt == CONVATTN_BF16 ? CALL(float, bf16_t) : CALL(float, float)))

template <typename TI, typename TO>
static hipError_t run_fwd(StArgs a, const void *q, const void *k, const void *v, const float *w, void *ws, void *o, float *m, float *l,
                          hipStream_t s) {
    a.c = static_cast<float *>(ws);
    a.mx = reinterpret_cast<float *>(static_cast<unsigned char *>(ws) + matrix_bytes(a));
    hipError_t e = launch_window<false, TI>(a, q, k, nullptr, nullptr, nullptr, nullptr, w, nullptr, s);
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)(a.p.B * a.p.H), (a.p.Nq + PM - 1) / PM);
    if (a.p.d <= 64) fwd_product_kernel<4, TI, TO><<<grid, PNT, 0, s>>>(a, (const TI *)v, (TO *)o, m, l);
    else fwd_product_kernel<8, TI, TO><<<grid, PNT, 0, s>>>(a, (const TI *)v, (TO *)o, m, l);
    return hipGetLastError();
}
hipError_t staged_fwd(const Problem &p, int in_dt, int out_dt, const void *q, const void *k, const void *v, const float *w, void *ws, void *o,
                      float *m, float *l, hipStream_t s) {
    const StArgs a = make_args(p);
#define CALL(TI, TO) run_fwd<TI, TO>(a, q, k, v, w, ws, o, m, l, s)
    return STAGED_IO(CALL);
#undef CALL
}

template <typename TI, typename TO>
static hipError_t run_bwd(StArgs a, const void *q, const void *k, const void *v, const void *d_o, const float *D, const float *lse,
                          const float *w, void *ws, void *dq, void *dk, void *dv, float *dw, hipStream_t s) {
    unsigned char *base = static_cast<unsigned char *>(ws);
    const size_t mb = matrix_bytes(a);
    a.c = reinterpret_cast<float *>(base);
    a.pm = reinterpret_cast<float *>(base + mb);
    a.ds = reinterpret_cast<float *>(base + 2 * mb);
    float *part = dw ? reinterpret_cast<float *>(base + 3 * mb) : nullptr;
    hipError_t e = launch_window<true, TI>(a, q, k, v, d_o, D, lse, w, part, s);
    if (e != hipSuccess) return e;
    e = set_max_lds_once<unwindow_kernel>((int)kLdsBytes);
    if (e != hipSuccess) return e;
    const unsigned BH = (unsigned)(a.p.B * a.p.H);
    const int n_tiles = (int)dw_tiles(a);
    unwindow_kernel<<<dim3(BH * n_tiles), NT, ((TT + a.p.pq) * win_lds(a.p, true).sst + a.p.c_q * win_stride(a.p.c_k)) * sizeof(float), s>>>(a, w);
    const int tiles = ((a.p.Nq > a.p.Nk ? a.p.Nq : a.p.Nk) + PM - 1) / PM, tap_blocks = (a.p.c_q * a.p.c_k + 63) / 64;
    const int sums = !dw ? 0 : tap_blocks < 65535 - tiles ? tap_blocks : 65535 - tiles;   // (tiles <= 65534, staged_ok)
    const dim3 grid(BH, (dq ? 1 : 0) + (dk ? 2 : 0), tiles + sums);
#define CALL(DB) \
    bwd_product_kernel<DB, TI, TO><<<grid, PNT, 0, s>>>(a, (const TI *)q, (const TI *)k, (const TI *)d_o, (TO *)dq, (TO *)dk, (TO *)dv, n_tiles, part, dw)
    if (a.p.d <= 64) CALL(4);
    else CALL(8);
#undef CALL
    return hipGetLastError();
}
hipError_t staged_bwd(const Problem &p, int in_dt, int out_dt, const void *q, const void *k, const void *v, const void *d_o, const float *D,
                      const float *lse, const float *w, void *ws, void *dq, void *dk, void *dv, float *dw, hipStream_t s) {
    const StArgs a = make_args(p);
#define CALL(TI, TO) run_bwd<TI, TO>(a, q, k, v, d_o, D, lse, w, ws, dq, dk, dv, dw, s)
    return STAGED_IO(CALL);
#undef CALL
}

}  // namespace convattn
