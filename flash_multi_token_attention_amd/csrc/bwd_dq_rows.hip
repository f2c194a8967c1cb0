// Launches of the dQ = dS K product (dq_rows.hpp).
#include "dq_rows.hpp"

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

}  // namespace convattn
