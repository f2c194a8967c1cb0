"""Autograd Function, module and functional form of head-mixing attention, with the reference's
names, constructor arguments and parameter name (head_conv_attn/head_conv_attn.py:11-115)."""
from __future__ import annotations

import math

import torch
import torch.nn as nn
from torch.autograd import Function

from .ops import backward, bwd_dkdv, bwd_dq_dw, forward


class HeadConvAttentionFunction(Function):
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
        grad_q = grad_k = grad_v = grad_w = None
        need_q, need_k, need_v, need_w = ctx.needs_input_grad[:4]
        if (need_q or need_w) and (need_k or need_v):
            lo = torch.bfloat16 if q.dtype == k.dtype == v.dtype == torch.bfloat16 else torch.float32
            grad_q, grad_k, grad_v, grad_w = backward(q, k, v, w, output, grad_output, l, m, causal=ctx.causal,
                                                      scale=ctx.scale, out_dtype=lo)
            return (grad_q.to(q.dtype), grad_k.to(k.dtype), grad_v.to(v.dtype), grad_w.to(w.dtype), None, None)
        if ctx.needs_input_grad[0] or ctx.needs_input_grad[3]:
            grad_q, grad_w = bwd_dq_dw(q, k, v, w, output, grad_output, l, m, causal=ctx.causal, scale=ctx.scale)
            grad_q, grad_w = grad_q.to(q.dtype), grad_w.to(w.dtype)
        if ctx.needs_input_grad[1] or ctx.needs_input_grad[2]:
            grad_k, grad_v = bwd_dkdv(q, k, v, w, output, grad_output, l, m, causal=ctx.causal, scale=ctx.scale)
            grad_k, grad_v = grad_k.to(k.dtype), grad_v.to(v.dtype)
        return grad_q, grad_k, grad_v, grad_w, None, None


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
