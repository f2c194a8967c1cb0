"""Window kernels on inputs with an infinity or NaN: the maximum of a row that sees an infinite score is +inf, and rows whose window does
not reach the value are what they are without it."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from tests.test_gpu_parity_mfma import _run_bwd
from tests.util import TOL_BF16, max_abs, oracle_bwd, oracle_fwd, rand_case, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# sparse and dense windows, odd and even tap slots, keys of a row tile in one workgroup and in several (N >= 1000)
@pytest.mark.parametrize("N,d,c_q,c_k,causal", [
    (200, 64, 6, 11, True), (200, 128, 8, 15, False), (200, 128, 11, 15, False), (200, 32, 7, 17, False), (1100, 64, 3, 3, True), (1100, 128, 6, 17, True),
])
def test_maximum_is_infinite(N, d, c_q, c_k, causal):
    Q, K, V, _, W = rand_case(1, 2, N, N, d, c_q, c_k, torch.bfloat16, seed=N + d)
    W = W.abs() + 0.05              # (one sign: no row adds +inf and -inf)
    key = 37
    Q[..., 0] = Q[..., 0].abs() + 0.5
    K[0, 0, key, 0] = 1.0           # the finite case, then infinite scores of this key in head 0
    args = (W.to(DEV), scale_of(d), c_q - 1, (c_k - 1) // 2, causal)
    _, M_fin, L_fin = ops.forward(Q.to(DEV), K.to(DEV), V.to(DEV), *args, out_dtype=torch.float32)
    _, M_ref, _ = oracle_fwd(Q, K, V, W, causal)
    assert max_abs(M_fin, M_ref) <= TOL_BF16
    K[0, 0, key, 0] = float("inf")
    _, M, L = ops.forward(Q.to(DEV), K.to(DEV), V.to(DEV), *args, out_dtype=torch.float32)
    # (the rows before the first have zeros for Q, whose product with the infinity is NaN: without the mask the first rows see one)
    first = key if causal else c_q - 1
    assert bool((M[0, 0, first:] == float("inf")).all()) and bool(L[0, 0, first:].isnan().all())
    assert torch.equal(M[0, 1], M_fin[0, 1]) and torch.equal(L[0, 1], L_fin[0, 1])
    if causal:
        assert max_abs(M[0, 0, :key], M_ref[0, 0, :key]) <= TOL_BF16 and bool(L[0, 0, :key].isfinite().all())


# each tap slot count as wide as it is: a narrower window has zero weights for older rows
@pytest.mark.parametrize("c_q,c_k", [(3, 3), (6, 11), (7, 7), (8, 9), (11, 11), (11, 17)])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("row", [100, 101])
def test_forward_rows_outside_the_window(c_q, c_k, d, row):
    N = 200
    Q, K, V, _, W = rand_case(1, 2, N, N, d, c_q, c_k, torch.bfloat16, seed=c_q + d)
    Q[:, :, row] = 0
    O_ref, M_ref, _ = oracle_fwd(Q, K, V, W, True)
    Q[:, :, row] = float("nan")
    O, M, _ = ops.forward(Q.to(DEV), K.to(DEV), V.to(DEV), W.to(DEV), scale_of(d), c_q - 1, (c_k - 1) // 2, True, out_dtype=torch.float32)
    assert bool(O[:, :, row:row + c_q].isnan().all())
    rows = [i for i in range(N) if not row <= i < row + c_q]
    assert max_abs(O[:, :, rows], O_ref[:, :, rows]) <= TOL_BF16 and max_abs(M[:, :, rows], M_ref[:, :, rows]) <= TOL_BF16


@pytest.mark.parametrize("c_q,c_k", [(3, 3), (6, 11), (8, 9), (11, 11)])
@pytest.mark.parametrize("d,causal", [(32, True), (64, False), (128, True)])
@pytest.mark.parametrize("row", [100, 101])
def test_backward_rows_outside_the_window(c_q, c_k, d, causal, row):
    N = 200
    Q, K, V, dO, W = rand_case(1, 2, N, N, d, c_q, c_k, torch.bfloat16, seed=c_q + d)
    dO[:, :, row] = 0
    want = oracle_bwd(Q, K, V, W, dO, causal)[0]
    dO[:, :, row] = float("nan")
    rows = [i for i in range(N) if not row - c_q < i <= row]   # (a dS row takes dC of its own row and of the c_q - 1 after it)
    for one_pass in (False, True):
        got = _run_bwd(*[t.to(DEV) for t in (Q, K, V, dO, W)], causal, torch.float32, one_pass)[0]
        assert max_abs(got[:, :, rows], want[:, :, rows]) <= TOL_BF16


# 7 taps have slots of their own up to d = 64
@pytest.mark.parametrize("d,causal", [(32, True), (32, False), (64, True), (64, False)])
@pytest.mark.parametrize("row", [100, 101])
def test_backward_rows_outside_a_window_of_seven(d, causal, row):
    test_backward_rows_outside_the_window(7, 7, d, causal, row)
