"""The window as sparse matrix products: every count of tap slots with the narrowest and the widest band such a product holds and, at 17 key
taps, the dense form, with weights of one size on all taps, against the CPU oracle."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from tests.test_gpu_parity_mfma import _run_bwd
from tests.util import TOL_BF16, TOL_DW_REL, max_abs, oracle_bwd, oracle_fwd, rand_case, rel_max, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("c_q", [1, 3, 5, 6, 7, 8, 10, 11])
@pytest.mark.parametrize("c_k", [1, 13, 15, 17])
@pytest.mark.parametrize("d,causal", [(32, False), (64, True), (128, True), (128, False)])
def test_window_forward(c_q, c_k, d, causal):
    N = 4 * (33 - c_q) + 2   # two rows beyond a tile of up to 11 query taps, two or three key steps of 32 and a remainder
    Q, K, V, _, W = rand_case(1, 2, N, N, d, c_q, c_k, torch.bfloat16, seed=c_q + c_k + d, w_mode="rand")
    W /= (c_q * c_k) ** 0.5   # (scores of the size of one tap's)
    O_ref, M_ref, L_ref = oracle_fwd(Q, K, V, W, causal)
    g = [t.to(DEV) for t in (Q, K, V, W)]
    assert ops.kernel_path(g[0], g[1], g[3], causal) == "mfma"
    O, M, L = ops.forward(*g, scale_of(d), c_q - 1, (c_k - 1) // 2, causal, out_dtype=torch.float32)
    assert max_abs(O, O_ref) <= TOL_BF16 and max_abs(M, M_ref) <= TOL_BF16 and rel_max(L, L_ref) <= TOL_BF16


@pytest.mark.parametrize("c_q", [1, 3, 5, 6, 7, 8, 11])
@pytest.mark.parametrize("c_k", [1, 13, 15])
@pytest.mark.parametrize("d,causal", [(32, True), (64, False), (128, True)])
def test_window_backward(c_q, c_k, d, causal):
    N = 161   # a row of a second key block's dK and dV, and of a sixth row tile
    Q, K, V, dO, W = rand_case(1, 2, N, N, d, c_q, c_k, torch.bfloat16, seed=c_q + c_k + d, w_mode="rand")
    W /= (c_q * c_k) ** 0.5
    ref = oracle_bwd(Q, K, V, W, dO, causal)
    got = _run_bwd(*[t.to(DEV) for t in (Q, K, V, dO, W)], causal, torch.float32, True)
    for a, b in zip(got[:3], ref[:3]):
        assert max_abs(a, b) <= TOL_BF16
    assert rel_max(got[3], ref[3]) <= TOL_DW_REL
