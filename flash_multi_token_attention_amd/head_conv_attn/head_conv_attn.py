"""Autograd Function, module and functional form of head-mixing attention, with the reference's
names, constructor arguments and parameter name (head_conv_attn/head_conv_attn.py:11-115)."""
from __future__ import annotations

import math

import torch
import torch.nn as nn
from torch.autograd import Function

from .. import _lib
from .ops import backward, bwd_dkdv, bwd_dq_dw, forward


def _backward(q, k, v, w, output, grad_output, l, m, causal, scale, want_q, want_kv):
    """[dq, dk, dv, dw] in the dtypes of their tensors, None for those not wanted."""
    gq = gk = gv = gw = None
    if want_q and want_kv:
        lo = torch.bfloat16 if q.dtype == k.dtype == v.dtype == torch.bfloat16 else torch.float32
        gq, gk, gv, gw = backward(q, k, v, w, output, grad_output, l, m, causal=causal, scale=scale, out_dtype=lo)
    elif want_q:
        gq, gw = bwd_dq_dw(q, k, v, w, output, grad_output, l, m, causal=causal, scale=scale)
    elif want_kv:
        gk, gv = bwd_dkdv(q, k, v, w, output, grad_output, l, m, causal=causal, scale=scale)
    return [None if g is None else g.to(t.dtype) for g, t in ((gq, q), (gk, k), (gv, v), (gw, w))]


_native = None


def _host():
    global _native
    if _native is None:
        h = _lib.host()
        h.set_slow_backward("mix", _backward)
        _native = h
    return _native


class HeadConvAttentionFunction(Function):
    """``apply`` runs the native host path (csrc/host.cpp) where it takes the call; ``forward`` and ``backward`` are
    what it does for everything else."""

    @classmethod
    def apply(cls, q, k, v, w, causal=False, scale=None):
        if cls is HeadConvAttentionFunction and all(isinstance(t, torch.Tensor) for t in (q, k, v, w)):
            out = _host().mix_attention(q, k, v, w, bool(causal), 1.0 / math.sqrt(q.shape[-1]) if scale is None else scale)
            if out is not None:
                return out
        return super().apply(q, k, v, w, causal, scale)

    @staticmethod
    def forward(ctx, q, k, v, w, causal=False, scale=None):
        if scale is None:
            scale = 1.0 / math.sqrt(q.shape[-1])
        output, l, m = forward(q, k, v, w, scale=scale, causal=causal)
        ctx.save_for_backward(q, k, v, w, output, l, m)
        ctx.causal = causal
        ctx.scale = scale
        return output

    @staticmethod
    def backward(ctx, grad_output):
        q, k, v, w, output, l, m = ctx.saved_tensors
        need_q, need_k, need_v, need_w = ctx.needs_input_grad[:4]
        return (*_backward(q, k, v, w, output, grad_output, l, m, ctx.causal, ctx.scale, need_q or need_w, need_k or need_v),
                None, None)


class HeadConvAttention(nn.Module):
    """Attention with a dense linear map across the head dimension before the softmax."""

    def __init__(self, n_heads, dtype=torch.float16):
        super().__init__()
        self.n_heads = n_heads
        self.dtype = dtype
        self.head_conv_weights = nn.Parameter(torch.randn(n_heads, n_heads, dtype=dtype) / math.sqrt(n_heads))

    def forward(self, q, k, v, causal=False, scale=None):
        return HeadConvAttentionFunction.apply(q, k, v, self.head_conv_weights, causal, scale)


def head_conv_attention(q, k, v, w, causal=False, scale=None):
    return HeadConvAttentionFunction.apply(q, k, v, w, causal, scale)


__all__ = ["HeadConvAttentionFunction", "HeadConvAttention", "head_conv_attention"]
