"""The mix of 32 heads as products of three bf16 parts: fp32's precision over a range of weights, and the infinities and NaN that the
fp32 products take."""
import math

import pytest
import torch

from oracle import head_conv_oracle as hc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
H = 32


@pytest.mark.parametrize("N,d,causal", [(16, 32, True), (33, 64, False), (250, 128, True), (321, 64, True)])
@pytest.mark.parametrize("spread", [0.0, 6.0])
def test_precision_of_the_scores(N, d, causal, spread):
    # one weight of every row is 2^spread and more above the others, so a row's largest score is its product up to rounding: log sum exp
    # against 64 bits within 2^-22 of sum |w S| (fp32: 2^-24 for the product, 2^-24 for a sum that the others barely move; without
    # the products of the lowest parts 2^-18 of a product are missing, 2^-19 on average)
    from flash_multi_token_attention_amd.head_conv_attn import ops
    g = torch.Generator().manual_seed(N + d)
    Q, K, V = (torch.randn(2, H, N, d, generator=g).to(torch.bfloat16) for _ in range(3))
    W = torch.randn(H, H, generator=g) * 2.0 ** -(spread + 8)
    W[torch.arange(H), torch.randperm(H, generator=g)] = 8.0 * (1 + torch.rand(H, generator=g))
    sc = 1.0 / math.sqrt(d)
    O, L, M = ops.forward(*(t.to(DEV) for t in (Q, K, V, W)), scale=sc, causal=causal)
    S = torch.matmul(Q.double(), K.double().transpose(-1, -2).contiguous()) * sc
    Z = torch.matmul(W.double(), S.reshape(2, H, N * N)).reshape(2, H, N, N)
    size = torch.matmul(W.double().abs(), S.abs().reshape(2, H, N * N)).reshape(2, H, N, N)
    if causal:
        Z = Z.masked_fill(torch.ones(N, N, dtype=torch.bool).triu(1), -math.inf)
    top = Z.argmax(-1, keepdim=True)
    err = (M.double().cpu() + L.double().cpu().log() - torch.logsumexp(Z, -1)).norm()
    assert float(err) <= 2.0 ** -22 * float(size.gather(-1, top).norm())


def inputs(N, d, positive):
    g = torch.Generator().manual_seed(N)
    Q, K, V, dO = (torch.randn(1, H, N, d, generator=g) for _ in range(4))
    Q[..., 0] = -Q[..., 0].abs() - 0.1
    W = torch.randn(H, H, generator=g) / math.sqrt(H)
    return [t.to(torch.bfloat16) for t in (Q, K, V, dO)], W.abs() if positive else W


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("N,d,key", [(40, 64, 7), (200, 32, 133), (97, 128, 96)])
def test_a_key_of_minus_infinity(N, d, key, causal):
    # scores of one key are -inf in every head that has it, so its weight is 0 and nothing else changes
    from flash_multi_token_attention_amd.head_conv_attn import ops
    (Q, K, V, dO), W = inputs(N, d, True)
    K[0, 3, key, 0] = math.inf
    sc = 1.0 / math.sqrt(d)
    q, k, v, do, w = (t.to(DEV) for t in (Q, K, V, dO, W))
    O, L, M = ops.forward(q, k, v, w, scale=sc, causal=causal)
    Or, Lr, Mr = hc.forward(Q.float(), K.float(), V.float(), W, causal, sc)
    assert float((O.float().cpu() - Or).abs().max()) <= 2e-2
    assert float(((L.cpu() - Lr).abs() / Lr).max()) <= 1e-3
    ref = hc.backward_autograd(Q.float(), K.float(), V.float(), W, dO.float(), causal, sc)
    got = ops.backward(q, k, v, w, O, do, L, M, causal=causal, scale=sc)
    for name, a, want in zip(("dK", "dV"), got[1:3], ref[1:3]):   # (0 x inf in dQ and dw)
        assert float((a.cpu() - want).abs().max()) <= 1e-2 * max(1.0, float(want.abs().max())), name


def test_an_infinite_weight_and_nan_stay_where_they_are():
    from flash_multi_token_attention_amd.head_conv_attn import ops
    N, d = 70, 64
    (Q, K, V, _), W = inputs(N, d, False)
    sc = 1.0 / math.sqrt(d)
    Or, _, _ = hc.forward(Q.float(), K.float(), V.float(), W, True, sc)
    W[5, 9] = math.inf          # head 5 alone
    O, L, M = ops.forward(*(t.to(DEV) for t in (Q, K, V, W)), scale=sc, causal=True)
    keep = torch.arange(H) != 5
    assert bool(O[:, 5].isnan().any()) and float((O.float().cpu() - Or)[:, keep].abs().max()) <= 2e-2
    W[5, 9] = 0.0
    Q[0, 2, 40, 1] = math.nan   # row 40 of all heads
    Or, _, _ = hc.forward(Q.float(), K.float(), V.float(), W, True, sc)
    O, L, M = ops.forward(*(t.to(DEV) for t in (Q, K, V, W)), scale=sc, causal=True)
    rows = torch.arange(N) != 40
    assert bool(O[:, :, 40].isnan().all()) and float((O.float().cpu() - Or)[:, :, rows].abs().max()) <= 2e-2
