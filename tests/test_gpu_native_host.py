"""The native host path (csrc/host.cpp) gives what the Python path gives, bit for bit: odd row counts, strided inputs, partial
gradients, other weight dtypes and a capped workspace (where its backward hands over to Python)."""
import pytest
import torch

from flash_multi_token_attention_amd.conv_attn import ops
from flash_multi_token_attention_amd.conv_attn.module import FlashConvAttentionCUDAFunction as ConvFn
from flash_multi_token_attention_amd.head_conv_attn.head_conv_attn import HeadConvAttentionFunction as MixFn
from tests.util import rand_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _PyConv(ConvFn):   # (a subclass runs the Python forward and backward)
    pass


class _PyMix(MixFn):
    pass


def _grads(fn, tensors, needs, dO, *rest):
    leaves = [t.detach().clone().requires_grad_(n) for t, n in zip(tensors, needs)]
    # (strided views of a leaf reach the op where the caller had them)
    args = [l.transpose(1, 2).contiguous().transpose(1, 2) if l.dim() == 4 else l for l in leaves]
    O = fn.apply(*args, *rest)
    O.backward(dO)
    return [O.detach()] + [l.grad for l in leaves]


def _same(a, b):
    return all((x is None) == (y is None) and (x is None or torch.equal(x, y)) for x, y in zip(a, b))


@pytest.mark.parametrize("needs", [(1, 1, 1, 1), (1, 0, 0, 0), (0, 1, 0, 0), (0, 0, 1, 1)])
@pytest.mark.parametrize("dtype,w_dtype,N,cap", [(torch.bfloat16, torch.float32, 37, None), (torch.bfloat16, torch.bfloat16, 150, None),
                                                 (torch.float32, torch.float32, 37, None), (torch.bfloat16, torch.float32, 90, "2048")])
def test_window_attention(dtype, w_dtype, N, cap, needs, monkeypatch):
    if cap:
        monkeypatch.setenv("CONVATTN_MAX_WORKSPACE_BYTES", cap)
    Q, K, V, dO, W = (t.to(DEV) for t in rand_case(1, 3, N, N, 64, 6, 11, dtype, seed=N))
    rest = (0.125, 5, 5, True)
    needs = [bool(n) for n in needs]
    assert _same(_grads(ConvFn, (Q, K, V, W.to(w_dtype)), needs, dO, *rest), _grads(_PyConv, (Q, K, V, W.to(w_dtype)), needs, dO, *rest))


@pytest.mark.parametrize("needs", [(1, 1, 1, 1), (1, 0, 0, 0), (0, 1, 1, 0)])
@pytest.mark.parametrize("cap", [None, "0"])
def test_head_mixing(needs, cap, monkeypatch):
    if cap:
        monkeypatch.setenv("CONVATTN_MAX_WORKSPACE_BYTES", cap)
    Q, K, V, dO, _ = (t.to(DEV) for t in rand_case(1, 16, 37, 37, 32, 1, 1, torch.bfloat16, seed=3))
    W = torch.randn(16, 16, generator=torch.Generator().manual_seed(1)).to(DEV) / 4
    needs = [bool(n) for n in needs]
    assert _same(_grads(MixFn, (Q, K, V, W), needs, dO, True, None), _grads(_PyMix, (Q, K, V, W), needs, dO, True, None))


def test_double_use_and_freed_graph():
    Q, K, V, dO, W = (t.to(DEV) for t in rand_case(1, 2, 40, 40, 64, 3, 3, torch.bfloat16, seed=1))
    q = Q.clone().requires_grad_(True)
    O = ConvFn.apply(q, K, V, W, 0.125, 2, 1, True)
    a, = torch.autograd.grad(O, q, dO, retain_graph=True)
    b, = torch.autograd.grad(O, q, dO)
    assert torch.equal(a, b)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(O, q, dO)
    O = ConvFn.apply(q, K, V, W, 0.125, 2, 1, True)
    K.add_(1.0)   # a saved tensor changed in place
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(O, q, dO)


def test_decode_matches_the_checked_path():
    Q, K, V, _, W = (t.to(DEV) for t in rand_case(2, 3, 6, 333, 64, 6, 11, torch.bfloat16, seed=2))
    ws = tuple(torch.empty(2, 3, 5, *s, dtype=torch.float32, device=DEV) for s in ((64,), (), ()))
    a = ops.decode(Q, K, V, W, 5, 0.125)                 # native
    b = ops.decode(Q, K, V, W, 5, 0.125, workspace=ws)   # Python
    assert all(torch.equal(x, y) for x, y in zip(a[:3], b[:3]))
    with pytest.raises(RuntimeError, match="must be contiguous"):
        ops.decode(Q, K, V.transpose(1, 2).contiguous().transpose(1, 2), W, 5, 0.125)
