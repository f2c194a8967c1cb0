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


@pytest.mark.parametrize("N,d,causal", [(33, 64, False), (250, 128, True), (321, 32, True)])
def test_precision_of_the_transposed_mix(N, d, causal):
    # Heads 2p and 2p + 1 have the same scores' weights, V and dO, so the same dZ; head 16 + p, whose own scores are 0 (Q = 0), takes their
    # difference: dS = a dZ - a (1 + e) dZ with e about 2^-13.  What a product is short of comes out 2^13 times as large: fp32's 2^-24
    # (of w scale, and of the sum) 2^-11 each, beside the 2^-9 that the bf16 of dS leaves, half of it in the norm; without the lowest
    # parts 2^-18 of a product are missing, 2^-19 on average, a sixty-fourth of dS.
    from flash_multi_token_attention_amd.head_conv_attn import ops
    g = torch.Generator().manual_seed(N + d)
    Q, K, V, dO = (torch.randn(2, H, N, d, generator=g).to(torch.bfloat16) for _ in range(4))
    Q[:, 16:] = 0
    V[:, 1::2], dO[:, 1::2] = V[:, ::2], dO[:, ::2]
    W = torch.zeros(H, H)
    W[::2, :16] = torch.randn(16, 16, generator=g) / 4
    W[1::2] = W[::2]
    p = torch.arange(16)
    W[2 * p, 16 + p] = 1 + torch.rand(16, generator=g)
    W[2 * p + 1, 16 + p] = -W[2 * p, 16 + p] * (1 + 2.0 ** -13 * (1 + torch.rand(16, generator=g)))
    sc = 1.0 / math.sqrt(d)
    q, k, v, do, w = (t.to(DEV) for t in (Q, K, V, dO, W))
    O, L, M = ops.forward(q, k, v, w, scale=sc, causal=causal)
    got = ops.backward(q, k, v, w, O, do, L, M, causal=causal, scale=sc)[0].double().cpu()[:, 16:]
    want, short = transposed_mix_dq(Q, K, V, dO, O.cpu(), W, sc, causal)
    assert float((got - want).norm()) <= 2.0 ** -8 * float(want.norm())
    assert float((short - want).norm()) > 2.0 ** -8 * float(want.norm())   # (two parts of w would fail)


def transposed_mix_dq(Q, K, V, dO, O, W, sc, causal):
    """dQ of heads 16.. in 64 bits, D from the O that was stored; with W and with its two highest bf16 parts."""
    Q, K, V, dO, O = (t.double() for t in (Q, K, V, dO, O))
    B, _, N, _ = Q.shape
    kt, vt = K.transpose(-1, -2).contiguous(), V.transpose(-1, -2).contiguous()
    Z = torch.matmul(W.double(), torch.matmul(Q, kt).mul(sc).reshape(B, H, N * N)).reshape(B, H, N, N)
    if causal:
        Z = Z.masked_fill(torch.ones(N, N, dtype=torch.bool).triu(1), -math.inf)
    dZ = torch.softmax(Z, -1) * (torch.matmul(dO, vt) - (dO * O).sum(-1, keepdim=True))
    ws = W * sc
    hi = ws.to(torch.bfloat16).float()
    two = hi + (ws - hi).to(torch.bfloat16).float()
    return [torch.matmul(torch.matmul(w.double().t()[16:], dZ.reshape(B, H, N * N)).reshape(B, 16, N, N), K[:, 16:])
            for w in (W.double() * sc, two)]


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
