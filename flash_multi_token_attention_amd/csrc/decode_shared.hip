// Decode step of conv-attention for query heads that share KV heads (gfx950).
//
// A workgroup takes HG = 4 or 2 query heads of one KV head together, so the K / V stream of the KV head is read once
// for all of them; its 4 waves walk their own shares of the keys, 64 per iteration, as in decode_stream.hip (scores by
// MFMA straight from the loaded K rows, an fp32 strip [head][tap row][16 carried + 64 keys] in LDS, K of the next
// iteration and V of this one in flight).
// With one K / V stream for four heads it is the arithmetic per key that binds, not the stream: the
// one-head kernel's window (one key per lane: 17 single LDS reads, 5 reads of weights and 17
// multiply-adds per tap row and head), its 64-lane maximum per head and P.V on the VALU (640 instructions
// per head and iteration) took three times as long as the loads.  Here
//   * a lane has HG consecutive keys of one head (64 / HG lanes per head, all heads at once): a tap row is
//     five LDS reads for HG x 11 multiply-adds, the weights are read once for HG keys, and the maximum
//     of all heads is four DPP rotations (one more exchange for HG = 2);
//   * P.V is a matrix product: a probability is the sum of three bf16 numbers (8 significant bits each,
//     split off exactly, so the product has fp32's 24), rows 4 * part + head of the A operand, and the V
//     rows turned in registers (byte permutes) are B: 16 MFMAs and 64 permutes for all heads;
//   * a lane's V rows are consecutive keys of one page: one page lookup;
//   * the workgroups of one round (two per CU) share all keys of the batch evenly, whatever the lengths of its entries
//     are: a workgroup's set-up and wind-down cost as much as three iterations, and with n_splits equal
//     parts per entry the round waited for the longest entry's.  A workgroup that meets the start of a stream does set-up and
//     wind-down twice, so the start counts as four tiles: without it the round waited for those workgroups
//     (B8 H32 H_kv8 N4348 d128 3x3 39.6 -> 33.2 us, B16 H32 H_kv8 N2254 d64 11x11 38.8 -> 34.9, B4 H32 H_kv8 N20000 d128
//     6x11 57.5 -> 52.5; 0 to 22 % over 100 shapes, 3 % on average with those of few keys, which go another way; 5 and 6 tiles
//     give the same within 0.2 %, 3 and 8 half a per cent less).
// B32 H32 H_kv8 N8192 d128 6x11, pages of 64, lengths drawn from a quarter to all of N (670 to 770 MB of K / V): the whole call with the
// merge 285 -> 136 to 142 us, this kernel about 134 of it (765 MB: 141 to 149 under the tracer).  No unit is full then (vector ALUs 22 %, LDS 19 %): each of the two waves per
// SIMD is a chain of scores, window, softmax and P.V.  H32 H_kv8 N8192 d128 11x11, B16, pages of 256: kernel 258 -> 86 us.
#include "mfma_common.hpp"

namespace convattn {
namespace {

constexpr int NW = 4;
constexpr int IT = 64;             // keys per wave iteration
constexpr int SROW = IT + 16 + 4;  // floats per strip row: 16 carried + 64 new, padded
constexpr int PROW = IT + 8;       // bf16 per row of probability parts
constexpr int kHead = 4;           // tiles that the start of a stream counts for in the even share

template <int ROR>
__device__ __forceinline__ float row_rot(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + ROR, 0xf, 0xf, true));
}
// reductions over the LPH lanes of a head (16 or 32)
template <int LPH>
__device__ __forceinline__ float head_max(float v) {
    v = fmaxf(v, row_rot<8>(v));
    v = fmaxf(v, row_rot<4>(v));
    v = fmaxf(v, row_rot<2>(v));
    v = fmaxf(v, row_rot<1>(v));
    if constexpr (LPH == 32) v = fmaxf(v, __shfl_xor(v, 16, kWave));
    return v;
}
template <int LPH>
__device__ __forceinline__ float head_sum(float v) {
    v += row_rot<8>(v);
    v += row_rot<4>(v);
    v += row_rot<2>(v);
    v += row_rot<1>(v);
    if constexpr (LPH == 32) v += __shfl_xor(v, 16, kWave);
    return v;
}
__device__ __forceinline__ float lane_value(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// c[i] += sum over TAPS columns of one strip row, for KPL consecutive keys; srow: the first key's column of tap -8
template <int TAPS, int KPL>
__device__ __forceinline__ void window_row(float (&c)[KPL], const float *srow, const float *wrow) {
    constexpr int OFF = 8 - (TAPS - 1) / 2, VN = KPL;      // reads of VN floats at multiples of VN
    constexpr int FIRST = OFF / VN * VN, N = (OFF + TAPS + KPL - 1 - FIRST + VN - 1) / VN * VN;
    typedef float vec __attribute__((ext_vector_type(VN)));
    float sv[N], wv[(TAPS + 3) / 4 * 4];
#pragma unroll
    for (int i = 0; i < N; i += VN) {
        const vec x = *reinterpret_cast<const vec *>(srow + FIRST + i);
#pragma unroll
        for (int e = 0; e < VN; ++e) sv[i + e] = x[e];
    }
#pragma unroll
    for (int i = 0; i < TAPS; i += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4 *>(wrow + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) wv[i + e] = x[e];
    }
    // (two sums of their own for each row, as in the kernel of unshared heads: one chain over the window, 121 terms for 11 x 11,
    // raised the error of O against 64 bits by a quarter)
    float even[KPL], odd[KPL];
#pragma unroll
    for (int t = 0; t < TAPS; ++t)
#pragma unroll
        for (int i = 0; i < KPL; ++i) {
            float &r = t & 1 ? odd[i] : even[i];
            r = t < 2 ? wv[t] * sv[OFF - FIRST + t + i] : fmaf(wv[t], sv[OFF - FIRST + t + i], r);
        }
#pragma unroll
    for (int i = 0; i < KPL; ++i) c[i] += even[i] + odd[i];
}

template <int D, int HG, bool WIDE>
struct Lds {   // byte offsets
    static constexpr int MG = WIDE ? HG : HG / 2, KS = D / 32;
    static constexpr int probs = 0;                                  // [NW][12][PROW] bf16
    static constexpr int pages = probs + NW * 12 * PROW * 2;         // [NW][2][8]
    static constexpr int ml = pages + NW * 2 * 8 * 4;                // [NW][HG][2]
    static constexpr int out = ml + NW * HG * 2 * 4;                 // [NW][HG][D]
    static constexpr int qf = out + NW * HG * D * 4;                 // [MG][KS][64] of 16 bytes
    static constexpr int weights = qf + MG * KS * 1024;              // [HG][c_q][20]
    static int bytes(int cq) { return weights + HG * cq * 20 * 4 + NW * HG * cq * SROW * 4; }
};

// WIDE: windows of 9 to 16 query taps, a head fills the 16 columns of a score MFMA; otherwise two heads do (8 each)
template <int D, bool PAGED, int HG, bool WIDE>
__global__ __launch_bounds__(NW * 64, 2) void decode_shared_kernel(
    Problem p, KvArgs kv, int parts, const bf16_t *__restrict__ Q, const bf16_t *__restrict__ K,
    const bf16_t *__restrict__ V, const float *__restrict__ W, float *__restrict__ O_part,
    float *__restrict__ M_part, float *__restrict__ L_part) {
    using L = Lds<D, HG, WIDE>;
    constexpr int KS = D / 32, MG = L::MG;
    constexpr int CPR = D / 8;         // 16-byte chunks per K / V row
    constexpr int VT = IT / (64 / CPR);   // V rows per lane: VT consecutive keys
    constexpr int SETS = 16 / CPR;     // key sets that share the 16 columns of a V fragment (d = 64: 2)
    constexpr int LPH = 64 / HG, KPL = HG;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane_id = threadIdx.x & 63;
    const int cq = p.c_q, ck = p.c_k, pk = p.pk;
    bf16_t *s_p = reinterpret_cast<bf16_t *>(lds + L::probs) + wave * 12 * PROW;
    int *s_pid = reinterpret_cast<int *>(lds + L::pages) + wave * 16;
    float *s_ml = reinterpret_cast<float *>(lds + L::ml), *s_o = reinterpret_cast<float *>(lds + L::out);
    float *s_w = reinterpret_cast<float *>(lds + L::weights);
    float *strip = s_w + HG * cq * 20 + wave * HG * cq * SROW;

    auto load16 = [](const bf16_t *src) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src)); };
    auto keys_of = [&](int b) {
        return __builtin_amdgcn_readfirstlane(kv.seq_lens ? min(max(kv.seq_lens[b], 0), p.Nk) : p.Nk);
    };
    auto tiles_of = [](int keys) { return max((keys + IT - 1) / IT, 1); };

    // This workgroup's share: `share` tiles of 64 keys of all streams (batch entry, group of HG heads) laid end to end,
    // cut at the streams' ends; its part of a stream is partial w - (workgroup of the stream's first tile) of the n_splits.
    // parts > 0 instead: every stream has its own workgroup (1) or `parts` of them with one tile per wave.
    const int w = blockIdx.x, groups = p.H / HG;
    // A workgroup that meets a stream's start goes through set-up and wind-down once more, so a stream counts as
    // `head` tiles and then its own (a part of head tiles only is an empty one).
    int b, grp, Nk, t0, t1, nt, share = 1, head = kHead;
    unsigned int pos = 0, end = 0, start = 0;   // tiles with the heads; start: the stream's first
    if (parts) {
        const int s = w / parts;
        b = s / groups; grp = s % groups;
        Nk = keys_of(b);
        nt = tiles_of(Nk);
        t0 = w % parts * NW;
        t1 = parts == 1 ? nt : min(nt, t0 + NW);
        if (t0 >= nt) return;
    } else {
        int longest = tiles_of(p.Nk);
        unsigned int total = (unsigned int)p.B * longest;
        if (kv.seq_lens) {
            int sum = 0, mx = 0;
            for (int i = lane_id; i < p.B; i += 64) {
                const int t = tiles_of(min(kv.seq_lens[i], p.Nk));
                sum += t;
                mx = max(mx, t);
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                sum += __shfl_xor(sum, o, kWave);
                mx = max(mx, __shfl_xor(mx, o, kWave));
            }
            total = __builtin_amdgcn_readfirstlane(sum);
            longest = __builtin_amdgcn_readfirstlane(mx);
        }
        // (a stream of n tiles meets at most ceil(n / share) + 1 workgroups; 4 tiles are one per wave)
        auto even_share = [&](unsigned int tiles, int most) {
            return max(max(NW, (int)((tiles * groups + gridDim.x - 1) / gridDim.x)), (most + p.n_splits - 2) / (p.n_splits - 1));
        };
        share = even_share(total, longest);
        // Streams of one length that the bare share divides: no workgroup meets two of them, and heads would only
        // unsettle that (B32 H16 H_kv8 N718 d128, two workgroups per stream: 25.8 us, with heads 28.5).
        if (total == (unsigned int)p.B * longest && longest % share == 0) {
            head = 0;
        } else {
            longest += head;
            total += (unsigned int)p.B * head;
            share = even_share(total, longest);
        }
        total *= groups;
        const unsigned long long first = (unsigned long long)w * share;
        if (first >= total) return;
        pos = (unsigned int)first;
        end = min(total, pos + share);
        b = 0;
        if (kv.seq_lens) {
            for (;; b += 64) {   // (pos < total: some entry contains it)
                const int mine = b + lane_id < p.B ? tiles_of(min(kv.seq_lens[b + lane_id], p.Nk)) + head : 0;
                int incl = mine;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(incl, o, kWave);
                    incl += lane_id >= o ? v : 0;
                }
                const unsigned long long found = __ballot(pos < start + (unsigned int)incl * groups);
                if (found) {
                    const int at = __builtin_ctzll(found);
                    b += at;
                    start += (unsigned int)__builtin_amdgcn_readlane(incl - mine, at) * groups;
                    break;
                }
                start += (unsigned int)__builtin_amdgcn_readlane(incl, 63) * groups;
            }
        } else {
            b = pos / (unsigned int)(longest * groups);
            start = (unsigned int)b * longest * groups;
        }
        Nk = keys_of(b);
        nt = tiles_of(Nk);
        grp = (pos - start) / (nt + head);
        start += (unsigned int)grp * (nt + head);
        t0 = max((int)(pos - start) - head, 0);
        t1 = min(nt, max((int)(end - start) - head, 0));
    }

    for (;;) {   // parts of streams
    int lane = lane_id;
    asm volatile("" : "+v"(lane));   // (no room in registers for everything that could be kept from part to part)
    const int g = lane >> 4, n = lane & 15, tid = wave * 64 + lane;
    const int cc = lane % CPR, gph = lane / CPR;   // this lane's V column chunk and run of keys
    const int hh_l = lane / LPH, kg = lane % LPH;  // this lane's head and its KPL keys in the window and the softmax
    const int row_head = WIDE ? 0 : (n >> 3), row_tap = WIDE ? n : (n & 7);
    const int h = grp * HG, hk = h / kv.group;   // first query head of the part
    const size_t bh = (size_t)b * p.H + h;
    const int sp = parts ? w % parts : w - (int)(start / share);
    const bf16_t *Kb = K + (PAGED ? 0 : b * p.kv_bstride) + hk * p.kv_hstride;
    const bf16_t *Vb = V + (PAGED ? 0 : b * p.kv_bstride) + hk * p.kv_hstride;
    // page numbers of the rows w0-8 .. w0+71 around an iteration (w0 a multiple of 64; at most 6 pages),
    // by scalar loads from the read-only table into slot (w0 / 64) & 1
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(4))) int *tbl_ptr_t;
#else
    typedef const int *tbl_ptr_t;
#endif
    tbl_ptr_t tbl = PAGED ? (tbl_ptr_t)(kv.table + (size_t)b * kv.table_stride) : (tbl_ptr_t) nullptr;
    auto fetch_pages = [&](int w0) {
        if constexpr (PAGED) {
            const int first = min(max(w0 - 8, 0), Nk - 1) >> kv.page_shift, last = (Nk - 1) >> kv.page_shift;
            int mine = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int id = tbl[min(first + i, last)];
                mine = lane == i ? id : mine;
            }
            if (lane < 8) s_pid[((w0 >> 6) & 1) * 8 + lane] = mine;
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
    };
    // row rr of [min(w0 - 8, Nk - 1), min(w0 + 71, Nk - 1)]
    auto row_ptr = [&](int w0, const bf16_t *base, int rr) -> const bf16_t * {
        if constexpr (PAGED) {
            const int first = min(max(w0 - 8, 0), Nk - 1) >> kv.page_shift;
            const int page = s_pid[((w0 >> 6) & 1) * 8 + (rr >> kv.page_shift) - first];
            return base + (size_t)page * kv.page_stride + (size_t)(rr & ((1 << kv.page_shift) - 1)) * D;
        } else {
            return base + (size_t)rr * D;
        }
    };

    // keys of this wave
    const int per_wave = (t1 - t0 + NW - 1) / NW;
    const int lo = (t0 + wave * per_wave) * IT, hi = min(Nk, min(t1, t0 + (wave + 1) * per_wave) * IT);

    u32x4 kfirst[KS], kreg[4][KS];
    // K of an iteration: keys j0+8 .. j0+71.  After the last iteration one row (of this iteration's) is loaded instead
    // of none: with the loads under a branch every wait for V would also wait for the K rows issued after it.
    auto load_k = [&](int j0, bool more) {
        const int last = min(Nk - 1, more ? Nk - 1 : j0 - 8);
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
            const bf16_t *src = row_ptr(j0, Kb, min(j0 + 8 + blk * 16 + n, last)) + g * 8;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) kreg[blk][ks] = load16(src + ks * 32);
        }
    };
    if (lo < hi) {   // the first K rows are under way while Q and the weights are staged
        fetch_pages(lo);
        const bf16_t *src = row_ptr(lo, Kb, min(max(lo - 8 + n, 0), Nk - 1)) + g * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kfirst[ks] = load16(src + ks * 32);
        load_k(lo, true);
    }

    // window weights times the scale [head][tap row][20]: key tap bb at column bb - pk + half of the fixed 11 or 17
    const int half = pk <= 5 ? 5 : 8;
    for (int i = tid; i < HG * cq * 20; i += NW * 64) {
        const int row = i / 20, bb = i - row * 20 - (half - pk);
        s_w[i] = (bb >= 0 && bb < ck) ? W[((size_t)h * cq + row) * ck + bb] * p.scale : 0.f;
    }
    // Q fragments, in LDS (there are no registers for them): tap row a reads resident row Nq - c_q + a (zeros if there is none)
    for (int i = wave; i < MG * KS; i += NW) {
        const int m = i / KS, ks = i % KS;
        const int ri = p.Nq - cq + row_tap, hh = (WIDE ? m : 2 * m) + row_head;
        u32x4 raw = {0u, 0u, 0u, 0u};
        if (row_tap < cq && ri >= 0)
            raw = *reinterpret_cast<const u32x4 *>(Q + ((bh + hh) * p.Nq + ri) * D + ks * 32 + g * 8);
        *reinterpret_cast<u32x4 *>(lds + L::qf + (i * 64 + lane) * 16) = raw;
    }
    auto q_at = [&](int m, int ks) -> bf16x8 {
        return *reinterpret_cast<const bf16x8 *>(lds + L::qf + ((m * KS + ks) * 64 + lane) * 16);
    };
    // Causal variant: tap row a sits at position Nk - c_q + a and sees no later key.
    const int row_pos = p.causal ? Nk - cq + row_tap : 0x7fffffff;

    f32x4 acc[SETS][8];
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[s][e] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m_run = kNegInf, l_run = 0.f;
    __syncthreads();

    // scores of 16 keys from key0 on -> strip columns col0 ..; edge: keys past the causal limit or outside [0, Nk) score zero
    auto scores = [&](const u32x4 (&kr)[KS], int key0, int col0, bool edge) {
        if constexpr (WIDE) asm volatile("" ::: "memory");   // (Q fragments of 4 heads are read again, not kept)
        f32x4 a4[MG];
#pragma unroll
        for (int m = 0; m < MG; ++m) a4[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int m = 0; m < MG; ++m) a4[m] = mfma_bf16(__builtin_bit_cast(bf16x8, kr[ks]), q_at(m, ks), a4[m]);
        if (row_tap < cq) {
#pragma unroll
            for (int m = 0; m < MG; ++m) {
                if (edge) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int key = key0 + 4 * g + r;
                        if (key > row_pos || key < 0 || key >= Nk) a4[m][r] = 0.f;
                    }
                }
                const int row = ((WIDE ? m : 2 * m) + row_head) * cq + row_tap;
                *reinterpret_cast<f32x4 *>(strip + row * SROW + col0 + 4 * g) = a4[m];
            }
        }
    };

    if (lo < hi) {
        scores(kfirst, lo - 8, 0, true);   // strip columns 0..15: keys lo-8 .. lo+7
        for (int j0 = lo; j0 < hi; j0 += IT) {
            // V of this iteration: keys j0 + gph * VT + t
            u32x4 vreg[VT];
            {
                const int r0 = min(j0 + gph * VT, Nk - 1);
                const bf16_t *src = row_ptr(j0, Vb, r0) + cc * 8;
                const unsigned int room = (unsigned int)(Nk - 1 - r0) * (D * 2);   // rows past the last one read the last one
#pragma unroll
                for (int t = 0; t < VT; ++t)
                    vreg[t] = load16(reinterpret_cast<const bf16_t *>(reinterpret_cast<const char *>(src) + min(t * D * 2u, room)));
            }
            fetch_pages(j0 + IT);

            const bool edge = j0 + IT + 8 > Nk - (p.causal ? cq : 0);
#pragma unroll
            for (int blk = 0; blk < 4; ++blk) scores(kreg[blk], j0 + 8 + blk * 16, 16 + blk * 16, edge);
            load_k(j0 + IT, j0 + IT < hi);
            __builtin_amdgcn_wave_barrier();

            // window: strip column of key x is x - (j0 - 8)
            float c[KPL];
#pragma unroll
            for (int i = 0; i < KPL; ++i) c[i] = 0.f;
            {
                const float *srow = strip + hh_l * cq * SROW + KPL * kg, *wrow = s_w + hh_l * cq * 20;
                if (half == 5) {
#pragma unroll 1
                    for (int a = 0; a < cq; ++a) window_row<11, KPL>(c, srow + a * SROW, wrow + a * 20);
                } else {
#pragma unroll 1
                    for (int a = 0; a < cq; ++a) window_row<17, KPL>(c, srow + a * SROW, wrow + a * 20);
                }
            }
            float mx = kNegInf;
#pragma unroll
            for (int i = 0; i < KPL; ++i) {
                if (j0 + KPL * kg + i >= hi) c[i] = kNegInf;
                mx = fmaxf(mx, c[i]);
            }
            // (key j0 exists, so the maximum is finite from the first iteration on)
            const float m_new = fmaxf(m_run, head_max<LPH>(mx));
            const float alpha = (m_run == kNegInf) ? 0.f : __expf(m_run - m_new);
            const bool moved = __any(m_new != m_run);
            m_run = m_new;
            l_run *= alpha;
            unsigned int part[3][KPL];
#pragma unroll
            for (int i = 0; i < KPL; ++i) {
                const float e = (c[i] == kNegInf) ? 0.f : __expf(c[i] - m_new);
                l_run += e;
                part[0][i] = __float_as_uint(e) & 0xffff0000u;
                const float r1 = e - __uint_as_float(part[0][i]);
                part[1][i] = __float_as_uint(r1) & 0xffff0000u;
                part[2][i] = __float_as_uint(r1 - __uint_as_float(part[1][i]));
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                typedef unsigned int pair_t __attribute__((ext_vector_type(KPL / 2), may_alias));
                pair_t two;
#pragma unroll
                for (int i = 0; i < KPL; i += 2) two[i / 2] = __builtin_amdgcn_perm(part[q][i + 1], part[q][i], 0x07060302u);
                *reinterpret_cast<pair_t *>(s_p + (4 * q + hh_l) * PROW + KPL * kg) = two;
            }
            __builtin_amdgcn_wave_barrier();
            // carry the last 16 score columns to the front for the next iteration
            for (int i = lane; i < HG * cq * 4; i += 64) {
                float *row = strip + (i >> 2) * SROW + 4 * (i & 3);
                *reinterpret_cast<f32x4 *>(row) = *reinterpret_cast<const f32x4 *>(row + IT);
            }
            if (moved) {
#pragma unroll
                for (int hh = 0; hh < HG; ++hh) {
                    const float a = lane_value(alpha, hh * LPH);
#pragma unroll
                    for (int s = 0; s < SETS; ++s)
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc[s][e][hh] *= a;
                }
            }
            // A: row 4 * part + head (rows from 12 on repeat row 11 and are not used), 8 keys of run SETS * g + s;
            // B: column cc * 8 + e.  The columns of a set's fragment that hold another set's keys are not used.
#pragma unroll
            for (int u = 0; u < VT / 8; ++u) {
                bf16x8 af[SETS];
#pragma unroll
                for (int s = 0; s < SETS; ++s)
                    af[s] = *reinterpret_cast<const bf16x8 *>(s_p + min(n, 11) * PROW + (SETS * g + s) * VT + 8 * u);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    u32x4 f;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        f[i] = __builtin_amdgcn_perm(vreg[8 * u + 2 * i + 1][e >> 1], vreg[8 * u + 2 * i][e >> 1],
                                                     (e & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
                    for (int s = 0; s < SETS; ++s) acc[s][e] = mfma_bf16(af[s], __builtin_bit_cast(bf16x8, f), acc[s][e]);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        l_run = head_sum<LPH>(l_run);
        // sum of the three parts (lanes g = 0..2) and, for d = 64, of the key sets (lanes n, n + 8)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
            for (int hh = 0; hh < HG; ++hh) {
                float v = acc[0][e][hh];
                if constexpr (SETS == 2) {
                    v = n < 8 ? v : acc[1][e][hh];
                    v += row_rot<8>(v);
                }
                v = g == 3 ? 0.f : v;
                v += __shfl_xor(v, 16, kWave);
                v += __shfl_xor(v, 32, kWave);
                if (lane < CPR) s_o[(wave * HG + hh) * D + cc * 8 + e] = v;
            }
        }
    }
    if (kg == 0) {
        s_ml[(wave * HG + hh_l) * 2] = m_run;
        s_ml[(wave * HG + hh_l) * 2 + 1] = l_run;
    }
    __syncthreads();
    // merge the 4 waves: o = sum o_w e^{m_w - m}, l = sum l_w e^{m_w - m}
    for (int i = tid; i < HG * D; i += NW * 64) {
        const int hh = i / D, col = i % D;
        float m = kNegInf;
#pragma unroll
        for (int w = 0; w < NW; ++w) m = fmaxf(m, s_ml[(w * HG + hh) * 2]);
        float o = 0.f, l = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float mw = s_ml[(w * HG + hh) * 2];
            if (mw != kNegInf) {
                o = fmaf(s_o[(w * HG + hh) * D + col], __expf(mw - m), o);
                l = fmaf(s_ml[(w * HG + hh) * 2 + 1], __expf(mw - m), l);
            }
        }
        const size_t slot = (bh + hh) * p.n_splits + sp;
        O_part[slot * D + col] = o;
        if (col == 0) {
            M_part[slot] = m;
            L_part[slot] = l;
        }
    }
    if (t1 == nt) {   // the stream's last part: the partials after it are empty
        const int empty = p.n_splits - 1 - sp;
        for (int i = tid; i < HG * empty; i += NW * 64) {
            const size_t slot = (bh + i / empty) * p.n_splits + sp + 1 + i % empty;
            M_part[slot] = kNegInf;
            L_part[slot] = 0.f;
        }
    }

    if (parts) {
        if (parts > 1) break;
        const long long next = (long long)b * groups + grp + gridDim.x;
        if (next >= (long long)p.B * groups) break;
        b = (int)(next / groups); grp = (int)(next % groups);
    } else {
        start += nt + head;
        if (start >= end) break;
        if (++grp == groups) { grp = 0; ++b; }
    }
    Nk = keys_of(b);
    nt = tiles_of(Nk);
    t0 = 0;
    t1 = parts ? nt : min(nt, max((int)(end - start) - head, 0));
    }
}

template <int D, bool PAGED, int HG, bool WIDE>
hipError_t launch(const Problem &p, const KvArgs &kv, const bf16_t *q, const bf16_t *k, const bf16_t *v, const float *w,
                  float *o_part, float *m_part, float *l_part, hipStream_t s) {
    using L = Lds<D, HG, WIDE>;
    hipError_t e = set_max_lds_once<decode_shared_kernel<D, PAGED, HG, WIDE>>(L::bytes(WIDE ? 16 : 8));
    if (e != hipSuccess) return e;
    // One round of workgroups: two per CU (their registers), one where the strips take more than half of the LDS.
    // Where four tiles per workgroup need no more of them than that, the streams are not laid end to end: an
    // even share would meet two streams, i.e. go through set-up and wind-down twice
    // (B1 H32 H_kv8 N700 d128: 28 against 17 us).
    const int most = 256 * (2 * L::bytes(p.c_q) <= (int)kLdsBytes ? 2 : 1), each = (p.Nk + NW * IT - 1) / (NW * IT);
    const long long streams = (long long)p.B * (p.H / HG), tiles = streams * ((p.Nk + IT - 1) / IT);
    const int parts = p.n_splits == 1 || tiles + kHead * streams > 0x7fffffffLL ? 1 : each <= p.n_splits && streams * each <= most ? each : 0;
    const long long wgs = parts > 1 ? streams * parts : parts ? streams : (tiles + NW - 1) / NW;
    decode_shared_kernel<D, PAGED, HG, WIDE><<<(int)(wgs < most ? wgs : most), NW * 64, L::bytes(p.c_q), s>>>(
        p, kv, parts, q, k, v, w, o_part, m_part, l_part);
    return hipGetLastError();
}
template <int D, bool PAGED>
hipError_t pick(const Problem &p, const KvArgs &kv, const bf16_t *q, const bf16_t *k, const bf16_t *v, const float *w,
                float *o_part, float *m_part, float *l_part, hipStream_t s) {
    const bool wide = p.c_q > 8;
    if (kv.group % 4 == 0)
        return wide ? launch<D, PAGED, 4, true>(p, kv, q, k, v, w, o_part, m_part, l_part, s)
                    : launch<D, PAGED, 4, false>(p, kv, q, k, v, w, o_part, m_part, l_part, s);
    return wide ? launch<D, PAGED, 2, true>(p, kv, q, k, v, w, o_part, m_part, l_part, s)
                : launch<D, PAGED, 2, false>(p, kv, q, k, v, w, o_part, m_part, l_part, s);
}

}  // namespace

// p.d is 64 or 128, kv.group is even
hipError_t decode_shared(const Problem &p, const KvArgs &kv, const void *q, const void *k, const void *v, const float *w,
                         float *o_part, float *m_part, float *l_part, hipStream_t s) {
    const bf16_t *Q = (const bf16_t *)q, *K = (const bf16_t *)k, *V = (const bf16_t *)v;
    if (p.d == 128)
        return kv.table ? pick<128, true>(p, kv, Q, K, V, w, o_part, m_part, l_part, s)
                        : pick<128, false>(p, kv, Q, K, V, w, o_part, m_part, l_part, s);
    return kv.table ? pick<64, true>(p, kv, Q, K, V, w, o_part, m_part, l_part, s)
                    : pick<64, false>(p, kv, Q, K, V, w, o_part, m_part, l_part, s);
}

}  // namespace convattn
