"""Staged fp32-arithmetic kernels (score-sized matrices in the workspace) at the edges of their 64 x 64 tiles and their
contraction steps, against the CPU oracle, and the kernels without that scratch which take over above the workspace cap."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from tests.util import TOL_BF16, TOL_DW_REL, TOL_FP32, max_abs, oracle_bwd, oracle_fwd, rand_case, rel_max, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # B, H, Nq, Nk, d, c_q, c_k, causal
    (1, 2, 63, 63, 64, 6, 11, True),
    (2, 1, 64, 64, 128, 11, 11, True),
    (1, 2, 129, 129, 64, 3, 3, True),
    (1, 1, 257, 257, 32, 7, 7, True),
    (1, 1, 193, 193, 72, 2, 13, True),
    (1, 2, 1, 1, 16, 6, 11, True),
    (1, 2, 65, 130, 64, 6, 11, False),
    (2, 1, 191, 62, 128, 9, 9, False),
    (1, 1, 70, 200, 24, 4, 17, False),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_staged_matches_oracle(case, dtype, monkeypatch):
    B, H, Nq, Nk, d, c_q, c_k, causal = case
    Q, K, V, dO, W = rand_case(B, H, Nq, Nk, d, c_q, c_k, dtype, seed=Nq + Nk + c_q, w_mode="rand")
    ref_o, ref = oracle_fwd(Q, K, V, W, causal), oracle_bwd(Q, K, V, W, dO, causal)
    g = [t.to(DEV) for t in (Q, K, V, dO, W)]
    win = (scale_of(d), c_q - 1, (c_k - 1) // 2, causal)
    tol, tol_w = (TOL_FP32, 1e-3) if dtype == torch.float32 else (TOL_BF16, TOL_DW_REL)
    for cap in (None, "1024"):
        if cap:
            monkeypatch.setenv("CONVATTN_MAX_WORKSPACE_BYTES", cap)
        O, M, L = ops.forward(g[0], g[1], g[2], g[4], *win, exact=True)
        assert max_abs(O, ref_o[0]) <= tol and max_abs(M, ref_o[1]) <= TOL_FP32 and rel_max(L, ref_o[2]) <= TOL_FP32
        D, LSE = ops.bwd_preprocess(O, g[3], M, L)
        dQ, dK, dV, dW = ops.backward(*g[:4], D, LSE, g[4], *win, exact=True)
        for name, got, want in (("dQ", dQ, ref[0]), ("dK", dK, ref[1]), ("dV", dV, ref[2])):
            assert max_abs(got, want) <= tol * max(1.0, float(want.abs().max())), name
        assert rel_max(dW, ref[3]) <= tol_w
