"""Shared-KV decode: the even share with a stream's start counted as tiles of its own.  256 streams over 512 workgroups, so that
workgroups meet two streams, end inside a stream's head (an empty part), or (12 tiles each) never meet two."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from oracle import conv_attn_oracle as orc
from tests.util import max_abs, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("Nk", [718, 780, 833])   # 12, 13 and 14 tiles
@pytest.mark.parametrize("lengths", ["none", "equal", "ragged", "one"])
@pytest.mark.parametrize("k_splits", [0, 3])
def test_shares(Nk, lengths, k_splits):
    B, H, H_kv, d, c_q, c_k = 64, 16, 4, 64, 3, 5
    g = torch.Generator().manual_seed(Nk)
    Q = torch.randn(B, H, c_q, d, generator=g).to(torch.bfloat16)
    K, V = (torch.randn(B, H_kv, Nk, d, generator=g).to(torch.bfloat16) for _ in range(2))
    W = 0.3 * torch.randn(H, c_q, c_k, generator=g)
    lens = [Nk] * B
    if lengths == "ragged":
        lens = [Nk] + torch.randint(1, Nk + 1, (B - 1,), generator=g).tolist()
    elif lengths == "one":      # entries of a tile between full ones: heads longer than their streams
        lens = [Nk if b % 3 == 0 else 1 + b for b in range(B)]
    seq = None if lengths == "none" else torch.tensor(lens, dtype=torch.int32, device=DEV)
    ref = orc.decode_kv(Q.float(), lambda b: K[b, :, :lens[b]].float(), lambda b: V[b, :, :lens[b]].float(), W, lens, scale_of(d), False)
    out = ops.decode_gqa(Q.to(DEV), K.to(DEV), V.to(DEV), W.to(DEV), k_splits, scale_of(d), False, seq_lens=seq)
    # fp32 arithmetic on both sides: terms of O and of the logarithm up to about 10, 1e-6 each from the scores' sums of 64 x 15
    assert max_abs(out[0], ref[0]) <= 1e-4
    assert max_abs(out[1] + torch.log(out[2]), ref[1] + torch.log(ref[2])) <= 1e-4
