"""Window forward in launches whose longer row tiles run at a higher wave priority: the bits of the same heads in launches that have
none."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# workgroups of the whole batch: 1.4 to 2 rounds of 768 (at most 2.1 - 3 / tiles of a head, which leaves two of these to the plain
# instance); of its parts less than one (and too few key steps to be split)
@pytest.mark.parametrize("d,c_q,c_k,B,H,N", [(64, 6, 11, 8, 16, 900), (64, 3, 3, 8, 16, 970), (32, 6, 11, 16, 16, 500), (64, 4, 5, 24, 12, 433),
                                             (32, 6, 11, 8, 16, 961), (64, 4, 5, 12, 11, 962), (32, 4, 3, 12, 16, 560)])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_same_bits(d, c_q, c_k, B, H, N, out):
    from flash_multi_token_attention_amd.conv_attn import ops
    rows = 4 * (33 - (3 if c_q <= 3 else 6))
    assert 1.4 * 768 < B * H * -(-N // rows) <= 2 * 768
    g = torch.Generator(device=DEV).manual_seed(N)
    Q, K, V = (torch.randn(B, H, N, d, generator=g, device=DEV, dtype=torch.bfloat16) for _ in range(3))
    W = 0.05 * torch.randn(H, c_q, c_k, generator=g, device=DEV)
    W[:, c_q - 1, c_k // 2] += 1
    win = (d ** -0.5, c_q - 1, c_k // 2, True)
    whole = ops.forward(Q, K, V, W, *win, out_dtype=out)
    for b in range(0, B, B // 4):
        part = [t[b:b + B // 4].contiguous() for t in (Q, K, V)]
        assert all(torch.equal(a[b:b + B // 4], c) for a, c in zip(whole, ops.forward(*part, W, *win, out_dtype=out)))
