"""Windows of 7 to 11 query taps: each instance of the window kernels by tap slots and head dimension, with lengths around the edges
of their row and key tiles, against the CPU oracle."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from tests.test_gpu_parity_mfma import _run_bwd
from tests.util import TOL_BF16, TOL_DW_REL, max_abs, oracle_bwd, oracle_fwd, rand_case, rel_max, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("c_q,c_k", [(7, 7), (8, 3), (9, 15), (10, 5), (11, 11)])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("N,causal", [(121, True), (159, False), (313, True)])
def test_tap_slots(c_q, c_k, d, N, causal):
    Q, K, V, dO, W = rand_case(1, 2, N, N, d, c_q, c_k, torch.bfloat16, seed=N + c_q + d)
    O_ref, M_ref, _ = oracle_fwd(Q, K, V, W, causal)
    ref = oracle_bwd(Q, K, V, W, dO, causal)
    g = [t.to(DEV) for t in (Q, K, V, dO, W)]
    O, M, _ = ops.forward(g[0], g[1], g[2], g[4], scale_of(d), c_q - 1, (c_k - 1) // 2, causal, out_dtype=torch.float32)
    assert max_abs(O, O_ref) <= TOL_BF16 and max_abs(M, M_ref) <= TOL_BF16
    for one_pass in (False, True):
        got = _run_bwd(*g, causal, torch.float32, one_pass)
        for a, b in zip(got[:3], ref[:3]):
            assert max_abs(a, b) <= TOL_BF16
        assert rel_max(got[3], ref[3]) <= TOL_DW_REL
