"""Shared-KV decode kernel: uneven lengths (even shares of all keys over the workgroups), tile edges, split counts that
bound the parts of a sequence, narrow and wide windows, against the CPU oracle."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from oracle import conv_attn_oracle as orc
from tests.util import max_abs, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("d,H,H_kv,c_q,c_k,page,k_splits", [
    (128, 8, 2, 6, 11, 16, 0), (128, 4, 2, 11, 11, 64, 0), (64, 8, 2, 11, 17, 16, 3), (64, 4, 2, 8, 3, 0, 0),
    (128, 8, 1, 3, 5, 0, 2), (128, 4, 1, 9, 13, 128, 1), (64, 16, 4, 6, 11, 16, 5),
])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("lens", [[1, 63, 64, 65, 300], [2500, 17, 1200], [1] * 40 + [129] * 30 + [257]])
def test_ragged(d, H, H_kv, c_q, c_k, page, k_splits, causal, lens):
    B, Nk = len(lens), max(lens)
    g = torch.Generator().manual_seed(d + H + c_q + B)
    Q = torch.randn(B, H, c_q, d, generator=g).to(torch.bfloat16)
    W = 0.3 * torch.randn(H, c_q, c_k, generator=g)
    sc = scale_of(d)
    lens_d = torch.tensor(lens, dtype=torch.int32, device=DEV)
    if page:
        n = -(-Nk // page)
        k_pool, v_pool = (torch.randn(B * n, H_kv, page, d, generator=g).to(torch.bfloat16) for _ in range(2))
        table = torch.randperm(B * n, generator=g).reshape(B, n).to(torch.int32)
        # rows past a sequence's end are never used, whatever they hold
        kp, vp = k_pool.to(DEV), v_pool.to(DEV)
        for b in range(B):
            if lens[b] % page:
                kp[table[b, lens[b] // page], :, lens[b] % page:] = float("nan")
                vp[table[b, lens[b] // page], :, lens[b] % page:] = float("nan")
        ref = orc.decode_kv(Q.float(), lambda b: orc.gather_paged(k_pool.float(), table, lens[b], b),
                            lambda b: orc.gather_paged(v_pool.float(), table, lens[b], b), W, lens, sc, causal)
        out = ops.decode_paged(Q.to(DEV), kp, vp, table.to(DEV), lens_d, Nk, W.to(DEV), k_splits, sc, causal)
    else:
        K, V = (torch.randn(B, H_kv, Nk, d, generator=g).to(torch.bfloat16) for _ in range(2))
        ref = orc.decode_kv(Q.float(), lambda b: K[b, :, :lens[b]].float(), lambda b: V[b, :, :lens[b]].float(), W, lens, sc,
                            causal)
        out = ops.decode_gqa(Q.to(DEV), K.to(DEV), V.to(DEV), W.to(DEV), min(k_splits, Nk), sc, causal, seq_lens=lens_d)
    assert max_abs(out[0], ref[0]) <= 1e-4
    assert max_abs(out[1] + torch.log(out[2]), ref[1] + torch.log(ref[2])) <= 1e-4
