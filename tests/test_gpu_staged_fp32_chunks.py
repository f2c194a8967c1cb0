"""Staged fp32 kernels at the edges of the 64 columns of Q and K that are staged at a time and of the contraction steps of 64, and
windows whose dW takes more sums than there are tiles; the products on their own give the same bits."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from tests.util import TOL_FP32, max_abs, oracle_bwd, oracle_fwd, rand_case, rel_max, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,H,Nq,Nk,d,c_q,c_k,causal", [
    (1, 2, 65, 65, 80, 6, 11, True), (1, 2, 128, 128, 112, 3, 3, True), (2, 1, 97, 97, 104, 7, 7, True),
    (1, 3, 161, 33, 120, 5, 5, False), (1, 2, 31, 190, 128, 11, 11, False), (3, 2, 20, 20, 64, 16, 15, True),
    (1, 1, 7, 7, 8, 16, 31, True), (2, 2, 192, 192, 64, 1, 1, True)])
def test_chunks_and_sums(B, H, Nq, Nk, d, c_q, c_k, causal):
    Q, K, V, dO, W = rand_case(B, H, Nq, Nk, d, c_q, c_k, torch.float32, seed=Nq + Nk + d, w_mode="rand")
    ref_o, ref = oracle_fwd(Q, K, V, W, causal), oracle_bwd(Q, K, V, W, dO, causal)
    q, k, v, do, w = (t.to(DEV) for t in (Q, K, V, dO, W))
    win = (scale_of(d), c_q - 1, (c_k - 1) // 2, causal)
    O, M, L = ops.forward(q, k, v, w, *win)
    # (the tolerances of the other tests of these kernels)
    assert max_abs(O, ref_o[0]) <= TOL_FP32 and max_abs(M, ref_o[1]) <= TOL_FP32 and rel_max(L, ref_o[2]) <= TOL_FP32
    D, LSE = ops.bwd_preprocess(O, do, M, L)
    args = (q, k, v, do, D, LSE, w, *win)
    got = ops.backward(*args)
    for name, a, want in zip(("dQ", "dK", "dV"), got, ref):
        assert max_abs(a, want) <= TOL_FP32 * max(1.0, float(want.abs().max())), name
    assert rel_max(got[3], ref[3]) <= 1e-3
    dQ, dW = ops.dq_backward(*args)
    assert torch.equal(dQ, got[0]) and torch.equal(dW, got[3])
    assert all(torch.equal(a, b) for a, b in zip(ops.dkdv_backward(*args), got[1:3]))
