"""Window kernels with weights that every output shows: a head for each corner tap of the window, with that tap alone at weight 1, and a
head with weights of one size on all taps.  Errors are taken relative to the size of each head's result, so that one missing or
misplaced weight is seen; that it would be is checked on the CPU, with one taken out of the oracle's."""
import ctypes
import functools

import pytest
import torch

from oracle import conv_attn_oracle as orc
from tests.test_gpu_parity_mfma import _run_bwd
from tests.util import oracle_bwd, oracle_fwd, rand_case, scale_of

DEV = "cuda:0"
NAMES = ("O", "dQ", "dK", "dV", "dW")
# bf16 rounding of P and dS (1e-3 of an element at the root mean square), fp16 rounding towards zero of scores of up to 32, whose last bit
# is 1/64 before the softmax scale (5e-4 of a probability at d = 64), and of dC (3e-4), fp16 weights (3e-4): about 2e-3 of a result's norm
TOL = 1e-2
N = 170   # five row tiles of 32 and 10 rows, one block of 128 keys and 42


@functools.lru_cache(maxsize=4)
def _case(c_q, c_k, d, B=1, rows=N):
    corners = [(0, 0), (0, c_k - 1), (c_q - 1, 0), (c_q - 1, c_k - 1)]
    Q, K, V, dO, W = rand_case(B, 5, rows, rows, d, c_q, c_k, torch.bfloat16, seed=c_q + c_k + d)
    W = torch.where(W >= 0, 1.0, -1.0) / (c_q * c_k) ** 0.5
    for h, (a, b) in enumerate(corners):
        W[h] = 0
        W[h, a, b] = 1
    return Q, K, V, dO, W


def _oracle(Q, K, V, dO, W, causal):
    return (oracle_fwd(Q, K, V, W, causal)[0],) + tuple(oracle_bwd(Q, K, V, W, dO, causal))


def _errors(got, want):
    """{name: [error of a head's result relative to its norm]}"""
    r = {}
    for name, a, b in zip(NAMES, got, want):
        dims = [i for i in range(b.dim()) if i != (0 if name == "dW" else 1)]
        a, b = a.double().cpu(), b.double()
        r[name] = ((a - b).square().sum(dims) / b.square().sum(dims)).sqrt()
    return r


WINDOWS = [(1, 15), (3, 3), (3, 13), (5, 1), (6, 11), (7, 7), (7, 15), (8, 15), (10, 13), (11, 15), (6, 17), (11, 17)]


@pytest.mark.gpu
@pytest.mark.parametrize("c_q,c_k", WINDOWS)
@pytest.mark.parametrize("d,causal", [(32, True), (64, False), (64, True), (128, True), (128, False)])
def test_every_tap(c_q, c_k, d, causal):
    Q, K, V, dO, W = _case(c_q, c_k, d)
    want = _oracle(Q, K, V, dO, W, causal)
    g = [t.to(DEV) for t in (Q, K, V, dO, W)]
    from flash_multi_token_attention_amd.conv_attn import ops
    O = ops.forward(g[0], g[1], g[2], g[4], scale_of(d), c_q - 1, (c_k - 1) // 2, causal, out_dtype=torch.float32)[0]
    for one_pass in (True, False):
        got = (O,) + tuple(_run_bwd(*g, causal, torch.float32, one_pass))
        for name, err in _errors(got, want).items():
            assert float(err.max()) <= TOL, (name, one_pass, err.tolist())


# few heads: workgroups that share the keys of a row tile (forward) and the rows of a key block (backward)
@pytest.mark.gpu
@pytest.mark.parametrize("c_q,c_k", [(3, 13), (6, 15), (6, 17), (8, 13), (11, 15)])
@pytest.mark.parametrize("d,causal", [(64, True), (128, True), (128, False)])
def test_every_tap_in_parts(c_q, c_k, d, causal):
    from flash_multi_token_attention_amd import _lib
    from flash_multi_token_attention_amd.conv_attn import ops
    Q, K, V, dO, W = _case(c_q, c_k, d, 1, 1050)
    g = [t.to(DEV) for t in (Q, K, V, dO, W)]
    lib, desc = _lib.load(), ops._desc(g[0], g[1], g[4], scale_of(d), causal, torch.float32)
    if c_q > 3:
        assert lib.convattn_fwd_split_workspace_bytes(ctypes.byref(desc)) > 0
    got = [ops.forward(g[0], g[1], g[2], g[4], scale_of(d), c_q - 1, (c_k - 1) // 2, causal, out_dtype=torch.float32)[0]]
    if c_k <= 15:
        assert lib.convattn_bwd_split_workspace_bytes(ctypes.byref(desc)) > lib.convattn_bwd_fused_workspace_bytes(ctypes.byref(desc))
        got += _run_bwd(*g, causal, torch.float32, True)
    for name, err in _errors(got, _oracle(Q, K, V, dO, W, causal)).items():
        assert float(err.max()) <= TOL, (name, err.tolist())


# 1.6 to 1.8 rounds of workgroups of three per CU: the longer tiles at a higher priority
@pytest.mark.gpu
@pytest.mark.parametrize("c_q,c_k", [(3, 13), (6, 15), (6, 17)])
def test_every_tap_long_tiles_first(c_q, c_k):
    from flash_multi_token_attention_amd.conv_attn import ops
    Q, K, V, _, W = _case(c_q, c_k, 64, 27, 1000)
    O = ops.forward(Q.to(DEV), K.to(DEV), V.to(DEV), W.to(DEV), scale_of(64), c_q - 1, (c_k - 1) // 2, True, out_dtype=torch.float32)[0]
    for b in (0, 26):
        want = oracle_fwd(Q[b:b + 1], K[b:b + 1], V[b:b + 1], W, True)[0]
        assert float(_errors([O[b:b + 1]], [want])["O"].max()) <= TOL


@pytest.mark.parametrize("c_q,c_k", WINDOWS)
@pytest.mark.parametrize("d,causal", [(64, False), (128, True)])
def test_a_missing_weight_shows(c_q, c_k, d, causal):
    """The least there is to be missed: one corner weight of the head that has all taps, in the convolution or in the transposed one alone."""
    Q, K, V, dO, W = _case(c_q, c_k, d)
    corners = sorted({(0, 0), (0, c_k - 1), (c_q - 1, 0), (c_q - 1, c_k - 1)})
    Q, K, V, dO = (t[:, 4:].float().expand(-1, len(corners), -1, -1) for t in (Q, K, V, dO))
    W = W[4:].expand(len(corners), -1, -1)
    less = W.clone()
    for h, (a, b) in enumerate(corners):
        less[h, a, b] = 0
    want = _oracle(Q, K, V, dO, W, causal)
    err = _errors(_oracle(Q, K, V, dO, less, causal), want)
    assert float(torch.stack([err["O"], err["dV"]]).min()) > 2 * TOL, err
    # the convolution with all of them, its gradient (the transposed one) without
    q, k = (t.clone().requires_grad_(True) for t in (Q, K))
    S = orc.masked_scores(q, k, scale_of(d), causal)
    C = orc.conv_scores(S, less)
    C = C + (orc.conv_scores(S, W) - C).detach()
    if causal:
        C = C.masked_fill(torch.ones(N, N, dtype=torch.bool).triu(1), float("-inf"))
    (torch.softmax(C, -1) @ V).backward(dO)
    err = _errors((want[0], q.grad, k.grad), want)
    assert float(torch.stack([err["dQ"], err["dK"]]).min()) > 2 * TOL, err
