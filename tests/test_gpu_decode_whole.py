"""Decode steps whose splits nobody sees: one workgroup per (batch, head) or fewer splits than asked for, against the CPU oracle and
against the step that returns its partials."""
import pytest
import torch

from flash_multi_token_attention_amd import _lib
from flash_multi_token_attention_amd.conv_attn import fwd_conv_attn_inference, ops
from oracle import conv_attn_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(B, H, r, Nk, d, c_q, c_k, seed):
    g = torch.Generator().manual_seed(seed)
    Q, K, V = (torch.randn(B, H, n, d, generator=g).to(torch.bfloat16) for n in (r, Nk, Nk))
    W = 0.05 * torch.randn(H, c_q, c_k, generator=g)
    W[:, c_q - 1, (c_k - 1) // 2] += 1.0
    return Q, K, V, W


# around a wave's 64 keys, four and eight waves of them
@pytest.mark.parametrize("Nk", [1, 63, 65, 257, 511, 512, 513, 1100])
@pytest.mark.parametrize("d,c_q,c_k,r", [(32, 3, 3, 16), (64, 7, 7, 16), (128, 6, 11, 6), (64, 16, 17, 5)])
@pytest.mark.parametrize("splits", [0, 1, 32])
def test_result_without_partials(Nk, d, c_q, c_k, r, splits):
    if splits > Nk:
        splits = Nk
    Q, K, V, W = _case(2, 3, r, Nk, d, c_q, c_k, seed=Nk + d)
    ref = orc.decode(Q.float(), K.float(), V.float(), W, d ** -0.5)
    q, k, v, w = (t.to(DEV) for t in (Q, K, V, W))
    got = fwd_conv_attn_inference(q, k, v, w, splits, d ** -0.5, c_q - 1, (c_k - 1) // 2, False)
    want = ops.decode(q, k, v, w, splits, d ** -0.5)[:3]
    for a, b, o in zip(got, want, ref):
        assert a.shape == b.shape and a.dtype == b.dtype
        # sums of at most 1100 fp32 terms in another order; the oracle's own products are rounded once more
        assert float((a - b).abs().max()) <= 1e-5 * max(1.0, float(b.abs().max()))
        assert float((a.cpu() - o).abs().max()) <= 2e-2 * max(1.0, float(o.abs().max()))
    bf = ops.decode_whole(q, k, v, w, splits, d ** -0.5, out_dtype=torch.bfloat16)
    assert bf[0].dtype == torch.bfloat16 and torch.equal(bf[0], got[0].to(torch.bfloat16))


def test_views_causal_and_refused_counts():
    Q, K, V, W = _case(2, 2, 6, 300, 64, 6, 11, seed=1)
    q, w = Q.to(DEV), W.to(DEV)
    room = torch.full((2, 2, 2, 512, 64), float("nan"), dtype=torch.bfloat16, device=DEV)   # (not to be read into the result)
    room[0, :, :, :300], room[1, :, :, :300] = K.to(DEV), V.to(DEV)
    k, v = room[0, :, :, :300], room[1, :, :, :300]
    for causal in (False, True):
        got = fwd_conv_attn_inference(q, k, v, w, 4, 0.125, 5, 5, causal)
        want = ops.decode(q, k, v, w, 4, 0.125, causal)[:3]
        assert all(float((a - b).abs().max()) <= 1e-5 * max(1.0, float(b.abs().max())) for a, b in zip(got, want))
    for bad in (-1, 301, 1025):
        with pytest.raises(RuntimeError, match="k_splits"):
            fwd_conv_attn_inference(q, k, v, w, bad, 0.125, 5, 5, False)


@pytest.mark.parametrize("Nk,splits", [(1, 1), (100, 32), (300, 3), (512, 32), (513, 4), (2048, 32), (2048, 1), (5000, 7), (40000, 700)])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_an_explicit_count_gives_a_head_the_same_bits_in_any_batch(Nk, splits, d):
    B, H = (4, 16) if Nk > 5000 else (24, 24)   # two workgroups fit a CU with d = 32: 576 heads are more than 512
    g = torch.Generator(device=DEV).manual_seed(Nk)
    splits = min(splits, Nk)
    Q, K, V = (torch.randn(B, H, n, d, generator=g, device=DEV, dtype=torch.bfloat16) for n in (6, Nk, Nk))
    W = 0.3 * torch.randn(H, 6, 11, generator=g, device=DEV)
    many = fwd_conv_attn_inference(Q, K, V, W, splits, d ** -0.5, 5, 5, False)
    for b, h in ((0, 1), (B - 1, 2)):
        few = fwd_conv_attn_inference(*(t[b:b + 1, :h].contiguous() for t in (Q, K, V)), W[:h].contiguous(), splits, d ** -0.5, 5, 5, False)
        assert all(torch.equal(a[b:b + 1, :h], c) for a, c in zip(many, few))


@pytest.mark.parametrize("Nk", [63, 300, 513, 2048])
@pytest.mark.parametrize("splits", [0, 1, 3, 32])
@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float32, 64), (torch.bfloat16, 40)])
def test_the_python_op_makes_the_same_step(Nk, splits, dtype, d, monkeypatch):
    # (where the native call declines: no host library, a dispatch mode)
    Q, K, V, W = (t.to(DEV) for t in _case(2, 3, 6, Nk, d, 6, 11, seed=Nk))
    Q, K, V = (t.to(dtype) for t in (Q, K, V))
    native = fwd_conv_attn_inference(Q, K, V, W, splits, d ** -0.5, 5, 5, False)
    monkeypatch.setattr(_lib, "host", lambda: None)
    plain = fwd_conv_attn_inference(Q, K, V, W, splits, d ** -0.5, 5, 5, False)
    assert all(a.dtype == b.dtype and torch.equal(a, b) for a, b in zip(native, plain))
    for bad in (-1, Nk + 1, 1025, 2 ** 32 + 1):
        with pytest.raises(RuntimeError, match="k_splits"):
            fwd_conv_attn_inference(Q, K, V, W, bad, d ** -0.5, 5, 5, False)
