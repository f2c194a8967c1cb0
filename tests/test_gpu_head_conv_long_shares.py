"""Head-mixing backward where a workgroup has many key steps (K and V asked for ahead, short tiles walked down): the gradients
of each batch entry are those of the entry alone, whose workgroups have few."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# steps per workgroup = B * (steps of the row tiles of 32 by keys of 16) / 256; the line is at 128, without the mask at 192
@pytest.mark.parametrize("B,N,causal", [(4, 2900, True), (4, 4096, True), (124, 497, True), (60, 515, False), (2, 3001, False),
                                        (90, 515, False), (4, 2501, False)])
def test_entries_of_long_shares(B, N, causal):
    from flash_multi_token_attention_amd.head_conv_attn import ops
    H, d, tiles = 16, 128, -(-N // 32)
    assert B * 2 * (tiles * (tiles + 1) // 2 if causal else tiles * tiles) > 128 * 256
    g = torch.Generator(device=DEV).manual_seed(N)
    q, k, v, do = (torch.randn(B, H, N, d, generator=g, device=DEV, dtype=torch.bfloat16) for _ in range(4))
    w = torch.randn(H, H, generator=g, device=DEV) / math.sqrt(H)
    kw = dict(causal=causal, scale=1.0 / math.sqrt(d))
    O, L, M = ops.forward(q, k, v, w, **kw)
    got = ops.backward(q, k, v, w, O, do, L, M, **kw)
    dw = torch.zeros(H, H, dtype=torch.float64, device=DEV)
    for b in range(B):
        one = [t[b:b + 1].contiguous() for t in (q, k, v, O, do, L, M)]
        want = ops.backward(*one[:3], w, *one[3:], **kw)
        # a (row, key) pair's P and dS do not depend on the order in which the keys are walked; dQ is summed over the keys in
        # another order where there are few row tiles (fp32 rounding, as dw)
        assert torch.equal(got[1][b:b + 1], want[1]) and torch.equal(got[2][b:b + 1], want[2]), b
        assert float((got[0][b:b + 1] - want[0]).norm() / want[0].norm()) <= 1e-5, b
        dw += want[3]
    # dw is summed over the steps of a workgroup in their order: fp32 rounding, as between groups of batch entries
    assert float((got[3] - dw).norm() / dw.norm()) <= 1e-5
