"""One-pass backward of head-mixing attention: block and tile edges, both gradient dtypes, and the kernels with O(N)
scratch that take over above the workspace cap."""
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
