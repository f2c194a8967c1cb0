// Launches of the dQ = dS K product (dq_rows.hpp).
#include "dq_rows.hpp"
#include "reduce_common.hpp"

namespace convattn {
namespace {

using namespace dq_rows;

template <int D, typename TO, bool KEYS>
__global__ __launch_bounds__(NW * 64) void dq_rows_kernel(Problem p, const bf16_t *__restrict__ K, const bf16_t *__restrict__ dS_ws,
                                                          const float *__restrict__ dc_scale, int n_kt, int n_rt,
                                                          int heads_inner, TO *__restrict__ dQ) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // (longest (causal) row tiles first)
    tile<D, TO, KEYS>(p, K, dS_ws, dc_scale, n_kt, n_rt, heads_inner, dQ, blockIdx.x, blockIdx.y, gridDim.z - 1 - blockIdx.z, smem);
}

template <int D, typename TO>
hipError_t launch(const Problem &p, const void *k, const void *ds_ws, const float *dc_scale, void *dq,
                  hipStream_t s, int heads_inner) {
    if (by_keys(p)) {
        constexpr int lds = lds_by_keys<D>;
        if (lds > 64 * 1024) {
            hipError_t e = set_max_lds_once<dq_rows_kernel<D, TO, true>>(lds);
            if (e != hipSuccess) return e;
        }
        dq_rows_kernel<D, TO, true><<<dim3(p.H, p.B, chain_row_tiles(p)), NW * 64, lds, s>>>(
            p, (const bf16_t *)k, (const bf16_t *)ds_ws, dc_scale, chain_key_tiles(p), chain_row_tiles(p), heads_inner, (TO *)dq);
        return hipGetLastError();
    }
    dq_rows_kernel<D, TO, false><<<dim3(p.H, p.B, (p.Nq + BQ - 1) / BQ), NW * 64, RowsLds<D>::total, s>>>(
        p, (const bf16_t *)k, (const bf16_t *)ds_ws, dc_scale, chain_key_tiles(p), chain_row_tiles(p), heads_inner, (TO *)dq);
    return hipGetLastError();
}

}  // namespace

hipError_t mfma_dq_from_rows(const Problem &p, int out_dt, const void *k, const void *ds_ws, const float *dc_scale,
                           void *dq, hipStream_t s, bool heads_inner) {
    if (p.d == 128) {
        if (out_dt == CONVATTN_BF16) return launch<128, bf16_t>(p, k, ds_ws, dc_scale, dq, s, heads_inner);
        return launch<128, float>(p, k, ds_ws, dc_scale, dq, s, heads_inner);
    }
    if (p.d == 32) {
        if (out_dt == CONVATTN_BF16) return launch<32, bf16_t>(p, k, ds_ws, dc_scale, dq, s, heads_inner);
        return launch<32, float>(p, k, ds_ws, dc_scale, dq, s, heads_inner);
    }
    if (out_dt == CONVATTN_BF16) return launch<64, bf16_t>(p, k, ds_ws, dc_scale, dq, s, heads_inner);
    return launch<64, float>(p, k, ds_ws, dc_scale, dq, s, heads_inner);
}

namespace {

// (256 threads; the first workgroups are dQ's, the longest tiles first)
template <int D, typename TO>
__global__ __launch_bounds__(NW * 64) void bwd_products_kernel(Problem p, const bf16_t *__restrict__ K, const bf16_t *__restrict__ dS_ws,
                                                               const float *__restrict__ dc_scale, int n_kt, int n_rt, int n_wg,
                                                               const float *__restrict__ dw_part, int share, int split_blocks,
                                                               const float *__restrict__ kv_part, TO *__restrict__ dQ,
                                                               TO *__restrict__ dK, TO *__restrict__ dV, float *__restrict__ dW) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int BH = p.B * p.H, ntap = p.c_q * p.c_k, n_dw = p.H * ((ntap + 63) / 64), i = blockIdx.x;
    if (i < BH * n_rt) {
        const int bh = i % BH;
        tile<D, TO, true>(p, K, dS_ws, dc_scale, n_kt, n_rt, 0, dQ, bh % p.H, bh / p.H, n_rt - 1 - i / BH, smem);
        return;
    }
    const int j = i - BH * n_rt;
    if (j < n_dw) {
        dw_reduce_block<NW * 64>(p.B, p.H, n_wg, ntap, dw_part, dW, j % p.H, j / p.H, reinterpret_cast<float (*)[64]>(smem));
        return;
    }
    constexpr int per = 2 * kKvKeysPerWg * D / 1024;
    const int r = j - n_dw, kb = r / per % split_blocks;
    chain_reduce_block(p, share, n_wg, kv_part, dK, dV, r % per, kb, r / per / split_blocks);
}
template <int D, typename TO>
hipError_t launch_products(const Problem &p, const void *k, const void *ds_ws, const float *dc_scale, int n_wg, const float *dw_part,
                           int share, const float *kv_part, void *dq, void *dk, void *dv, float *dw, hipStream_t s) {
    constexpr int lds = lds_by_keys<D>;
    static_assert(lds >= kDwChains * 64 * 4, "room for the dW chains");
    hipError_t e = set_max_lds_once<bwd_products_kernel<D, TO>>(lds);
    if (e != hipSuccess) return e;
    const int BH = p.B * p.H, n_rt = chain_row_tiles(p), split = share ? chain_split_blocks(p, share) : 0;
    const int grid = BH * n_rt + p.H * ((p.c_q * p.c_k + 63) / 64) + BH * split * (2 * kKvKeysPerWg * D / 1024);
    bwd_products_kernel<D, TO><<<grid, NW * 64, lds, s>>>(p, (const bf16_t *)k, (const bf16_t *)ds_ws, dc_scale, chain_key_tiles(p), n_rt,
                                                         n_wg, dw_part, share, split, kv_part, (TO *)dq, (TO *)dk, (TO *)dv, dw);
    return hipGetLastError();
}

}  // namespace

hipError_t mfma_bwd_products(const Problem &p, int out_dt, const void *k, const void *ds_ws, const float *dc_scale, int n_wg,
                             const float *dw_part, int share, const float *kv_part, void *dq, void *dk, void *dv, float *dw,
                             hipStream_t s) {
    if (by_keys(p)) {
#define CALL(DD) (out_dt == CONVATTN_BF16                                                                                          \
                      ? launch_products<DD, bf16_t>(p, k, ds_ws, dc_scale, n_wg, dw_part, share, kv_part, dq, dk, dv, dw, s)       \
                      : launch_products<DD, float>(p, k, ds_ws, dc_scale, n_wg, dw_part, share, kv_part, dq, dk, dv, dw, s))
        return p.d == 128 ? CALL(128) : p.d == 64 ? CALL(64) : CALL(32);
#undef CALL
    }
    hipError_t e = share ? chain_reduce(p, out_dt, share, kv_part, dk, dv, s) : hipSuccess;
    if (e == hipSuccess) e = mfma_dq_from_rows(p, out_dt, k, ds_ws, dc_scale, dq, s);
    if (e == hipSuccess) e = dw_reduce(p, n_wg, dw_part, dw, s);
    return e;
}

}  // namespace convattn
