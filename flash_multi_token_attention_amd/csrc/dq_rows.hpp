// dQ = dS K on bf16 MFMA (gfx950), second step of the one-pass backwards (launched by bwd_dq_rows.hip and, beside the
// head-mixing dK / dV product of small problems, by headmix_scores.hip).
//
// dS comes from the key-stationary kernel as bf16 blocks [key tile of 32][row tile of 32] of
// 32 rows x 32 keys, laid out [row parity][key half][row pair][16 keys] (the order in which that
// kernel's lanes hold it: each of its stores and each load here covers whole 128-byte lines; the
// softmax scale and the dC scale are already in it).  Workgroup
// = 4 waves = 128 query rows of one (batch, head); wave w owns rows i0 + 32w .. +31 and all D
// columns.  The product is dQ^T[d][row] += K^T[d][key] dS^T[key][row]: 16 bytes of a block are 8
// keys of one row, which is the B operand of a lane as it lies in memory, so dS goes from global
// memory straight into the MFMA operand registers (every block is read once, by one wave, in
// whole 1 KB pieces).  Only K passes through LDS (row-major, read with transpose reads), staged
// per step of 64 keys in two buffers with one barrier per step; the loads of the next two steps
// are in flight during the MFMAs.  Blocks the first kernel never wrote (key tile entirely after
// the row tile under the causal mask, or past the last key or row) are not read.
#pragma once
#include "mfma_common.hpp"

namespace convattn {
namespace dq_rows {

constexpr int NW = 4;
constexpr int BQ = 128;   // rows per workgroup
constexpr int BKS = 64;   // keys per step
constexpr int BLK = kChainKeys * kChainRows;  // elements per dS block

template <int D> struct RowsLds {
    static constexpr int RST = D * 2 + 16;
    static constexpr int k_bytes = BKS * RST;
    static constexpr int total = 2 * k_bytes;
};

// KEYS: the four waves of a workgroup share 32 rows, wave w takes the key steps w, w + 4, .. through LDS room of its own, and
// their sums are added at the end: for launches that would leave CUs idle or end with a few long workgroups.
// (B1 H8 N2048 d64 27.8 -> 14.8 us, B2 H8 N1531 22.6 -> 15.3, B1 H8 N1000 d128 19.2 -> 11.6.)
template <int D, typename TO, bool KEYS>
__device__ __forceinline__ void tile(const Problem &p, const bf16_t *__restrict__ K, const bf16_t *__restrict__ dS_ws,
                                     const float *__restrict__ dc_scale, int n_kt, int n_rt, int heads_inner,
                                     TO *__restrict__ dQ, int h, int b, int qt, unsigned char *smem) {
    using Lds = RowsLds<D>;
    constexpr int RST = Lds::RST;
    constexpr int DB = D / 16, CPR = D / 8;
    constexpr int K_CH = BKS * CPR;                 // 16-byte chunks of a K step
    constexpr int K_LD = K_CH / (KEYS ? 64 : NW * 64);   // per lane
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, n = lane & 15;
    const int i0 = qt * (KEYS ? kChainRows : BQ), rw = KEYS ? i0 : i0 + wave * 32, rt = rw / kChainRows;
    const int s0 = KEYS ? wave : 0, ds = KEYS ? NW : 1;   // this wave's first step and stride
    const bool causal = p.causal != 0;
    const size_t bh = (size_t)b * p.H + h;
    const bf16_t *Kb = K + bh * p.Nk * D;
    const size_t n_blk = (size_t)chain_ds_block_off(causal, n_rt, n_kt);
    const bf16_t *ws = dS_ws + (heads_inner ? b * n_blk * p.H + h : bh * n_blk) * BLK;
    const int blk_step = heads_inner ? p.H * BLK : BLK;   // elements from block to block

    f32x4 acc[2][DB];
#pragma unroll
    for (int ob = 0; ob < 2; ++ob)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[ob][db] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int k_end = causal ? min(p.Nk, i0 + (KEYS ? kChainRows : BQ)) : p.Nk;
    const int n_steps = (k_end + BKS - 1) / BKS;
    const bool row_ok = rt < n_rt;

    // the dS loads of steps s+1 and s+2 (two register sets) and the K loads of step s+1 (K comes from the
    // L2, which the other row tiles of the head keep it in) are in flight while step s is multiplied
    u32x4 kr[K_LD], sr_a[2][2], sr_b[2][2];
    auto load_k = [&](int s) {
#pragma unroll
        for (int i = 0; i < K_LD; ++i) {
            const int c = KEYS ? lane + i * 64 : tid + i * NW * 64, row = c / CPR, cc = c % CPR;
            kr[i] = load_row16_clamped<D>(Kb, s * BKS + row, p.Nk, cc * 8);
        }
    };
    auto load_ds = [&](int s, u32x4 (&sr)[2][2]) {
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
            const int kt = s * 2 + kp;
            // (a block that does not exist: any block that does; the registers are cleared before their use)
            const int rt_c = min(rt, n_rt - 1), kt_c = causal ? min(kt, rt_c) : min(kt, n_kt - 1);
            const size_t blk = (size_t)chain_ds_block_off(causal, n_rt, kt_c) + rt_c - chain_ds_first_rt(causal, kt_c);
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) {
                // every dS block is read once: non-temporal, so that it does not push K out of the caches.
                // Raw: blocks that do not exist are cleared where the registers are used (a select here
                // would wait for the load within this step)
                sr[kp][ob] = __builtin_nontemporal_load(
                    reinterpret_cast<const u32x4 *>(ws + blk * blk_step + ((ob * 2 + (g >> 1)) * 16 + n) * 16 + 8 * (g & 1)));
            }
        }
    };

    auto run_step = [&](int s, u32x4 (&sr)[2][2]) {
        unsigned char *Ks = smem + (KEYS ? wave : s & 1) * Lds::k_bytes;
#pragma unroll
        for (int i = 0; i < K_LD; ++i) {
            const int c = KEYS ? lane + i * 64 : tid + i * NW * 64, row = c / CPR, cc = c % CPR;
            *reinterpret_cast<u32x4 *>(Ks + row * RST + cc * 16) = zero_unless(s * BKS + row < p.Nk, kr[i]);
        }
        bf16x8 sf[2][2];
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
            const int kt = s * 2 + kp;
            // the block exists when its first key is a key and (causal) not after the tile's last row
            const bool ok = row_ok && kt * kChainKeys < p.Nk && (!causal || kt * kChainKeys <= rw + 31);
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) sf[kp][ob] = __builtin_bit_cast(bf16x8, zero_unless(ok, sr[kp][ob]));
        }
        if constexpr (KEYS) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
        load_k(s + ds);
        load_ds(s + 2 * ds, sr);
        if (causal && s * BKS > rw + 31) return;  // every key of the step is after the wave's rows

#pragma unroll
        for (int kp = 0; kp < BKS / 32; ++kp) {
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                // k slot 8g+e = key 8g+e of the 32-key tile, as in the dS rows
                bf16x4 lo = lds_read_tr4x16(Ks, RST, kp * 32 + 8 * g, db * 16, n);
                bf16x4 hi = lds_read_tr4x16(Ks, RST, kp * 32 + 8 * g + 4, db * 16, n);
                const bf16x8 kf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int ob = 0; ob < 2; ++ob) acc[ob][db] = mfma_bf16(kf, sf[kp][ob], acc[ob][db]);
            }
        }
    };
    load_k(s0);
    load_ds(s0, sr_a);
    load_ds(s0 + ds, sr_b);
    for (int s = s0; s < n_steps; s += 2 * ds) {
        run_step(s, sr_a);
        if constexpr (KEYS) {   // (this wave's reads of its room before its next writes)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
        if (s + ds < n_steps) run_step(s + ds, sr_b);
        if constexpr (KEYS) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
    }
    if constexpr (KEYS) {
        static_assert(2 * DB * 1024 <= Lds::k_bytes, "a wave's sums fit its room");
        f32x4 *mine = reinterpret_cast<f32x4 *>(smem + wave * Lds::k_bytes);
#pragma unroll
        for (int e = 0; e < 2 * DB; ++e) mine[e * 64 + lane] = acc[e / DB][e % DB];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 2 * DB; ++e) {
            if (e % NW != wave) continue;
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < NW; ++w) v += reinterpret_cast<const f32x4 *>(smem + w * Lds::k_bytes)[e * 64 + lane];
            acc[e / DB][e % DB] = v;
        }
    }

    // lane n of block ob = row 2 n + ob of the wave's 32; 4 consecutive head-dim columns per block
    const float inv = dc_scale ? 1.f / dc_scale[2 * bh] : 1.f;
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
        const int qpos = rw + 2 * n + ob;
        if (qpos < p.Nq) {
            TO *orow = dQ + (bh * p.Nq + qpos) * D;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                if (KEYS && (ob * DB + db) % NW != wave) continue;
                const int col = db * 16 + 4 * g;
                if constexpr (sizeof(TO) == 2) {
                    bf16x4 ov;
#pragma unroll
                    for (int r = 0; r < 4; ++r) ov[r] = (bf16_t)(acc[ob][db][r] * inv);
                    *reinterpret_cast<bf16x4 *>(orow + col) = ov;
                } else {
                    *reinterpret_cast<f32x4 *>(orow + col) = acc[ob][db] * inv;
                }
            }
        }
    }
}

// Whether the waves share the keys: with two workgroups per CU or fewer the launch is as long as its longest workgroup.
// (Not from 8192 rows on: a head's results do not depend on how many others there are.)
inline bool by_keys(const Problem &p) { return (long long)p.B * p.H * ((p.Nq + BQ - 1) / BQ) <= 512 && p.Nq < 8192; }
template <int D> constexpr int lds_by_keys = NW * RowsLds<D>::k_bytes;

}  // namespace dq_rows
}  // namespace convattn
