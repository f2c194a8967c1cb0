"""Head-mixing kernels with score-sized workspaces: block and tile edges, both gradient dtypes, score ranges beyond the
forward's fixed references, and the kernels with no or O(N) scratch that take over above the workspace cap."""
import math

import pytest
import torch

from oracle import head_conv_oracle as hc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,N,d", [(1, 16, 15, 128), (2, 16, 33, 64), (1, 16, 289, 128), (1, 32, 31, 128), (2, 32, 49, 64),
                                     (1, 32, 160, 32)])
def test_one_pass_backward(B, H, N, d, causal, monkeypatch):
    from flash_multi_token_attention_amd.head_conv_attn import ops
    g = torch.Generator().manual_seed(N * 3 + H)
    Q, K, V, dO = (torch.randn(B, H, N, d, generator=g).to(torch.bfloat16) for _ in range(4))
    W = torch.randn(H, H, generator=g) / math.sqrt(H)
    sc = 1.0 / math.sqrt(d)
    q, k, v, w, do = (t.to(DEV) for t in (Q, K, V, W, dO))
    O, L, M = ops.forward(q, k, v, w, scale=sc, causal=causal)
    ref = hc.backward_autograd(Q.float(), K.float(), V.float(), W, dO.float(), causal, sc)
    got = ops.backward(q, k, v, w, O, do, L, M, causal=causal, scale=sc)
    for name, a, want in zip(("dQ", "dK", "dV", "dW"), got, ref):
        assert float((a.cpu() - want).abs().max()) <= 1e-2 * max(1.0, float(want.abs().max())), name
    # bf16 gradients are the fp32 ones rounded; the partial passes compute the same tiles
    lo = ops.backward(q, k, v, w, O, do, L, M, causal=causal, scale=sc, out_dtype=torch.bfloat16)
    assert all(torch.equal(a.to(torch.bfloat16), b) for a, b in zip(got[:3], lo[:3])) and torch.equal(got[3], lo[3])
    dQ, dW = ops.bwd_dq_dw(q, k, v, w, O, do, L, M, causal=causal, scale=sc)
    dK, dV = ops.bwd_dkdv(q, k, v, w, O, do, L, M, causal=causal, scale=sc)
    assert all(torch.equal(a, b) for a, b in zip(got, (dQ, dK, dV, dW)))
    monkeypatch.setenv("CONVATTN_MAX_WORKSPACE_BYTES", "0")
    low = ops.backward(q, k, v, w, O, do, L, M, causal=causal, scale=sc)
    for name, a, want in zip(("dQ", "dK", "dV", "dW"), low, ref):
        assert float((a.cpu() - want).abs().max()) <= 1e-2 * max(1.0, float(want.abs().max())), name


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,N,d", [(16, 33, 128), (16, 300, 64), (32, 95, 128), (32, 130, 32)])
@pytest.mark.parametrize("grow", [0.0, 1.0, 6.0])
def test_forward_score_ranges(H, N, d, causal, grow, monkeypatch):
    # keys that grow along the sequence: the largest scores exceed those of the first tile of keys, from which the
    # forward takes a row's reference, by more than it allows for (60 in log2 units), more than once
    from flash_multi_token_attention_amd.head_conv_attn import ops
    g = torch.Generator().manual_seed(N + H)
    Q, K, V = (torch.randn(2, H, N, d, generator=g) for _ in range(3))
    K = K * (1.0 + grow * torch.arange(N).view(-1, 1) / 16)
    Q, K, V = (t.to(torch.bfloat16) for t in (Q, K, V))
    W = torch.randn(H, H, generator=g) / math.sqrt(H)
    sc = 1.0 / math.sqrt(d)
    args = [t.to(DEV) for t in (Q, K, V, W)]
    Or, Lr, Mr = hc.forward(Q.float(), K.float(), V.float(), W, causal, sc)
    for cap in (None, "0"):
        if cap is not None:
            monkeypatch.setenv("CONVATTN_MAX_WORKSPACE_BYTES", cap)
        O, L, M = ops.forward(*args, scale=sc, causal=causal)
        assert float((O.float().cpu() - Or).abs().max()) <= 2e-2
        assert float((M.cpu() - Mr).abs().max()) <= 1e-3 * max(1.0, 1e-2 * float(Mr.abs().max()))
        assert float(((L.cpu() - Lr).abs() / Lr).max()) <= 1e-3
