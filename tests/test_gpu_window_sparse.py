"""The window as sparse matrix products: every count of tap slots with the narrowest and the widest band such a product holds and, at 17 key
taps, the dense form, with weights of one size on all taps, against the CPU oracle."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from tests.util import TOL_BF16, max_abs, oracle_fwd, rand_case, rel_max, scale_of

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
