"""The attention half of a decoder block, x + out_proj(attention(norm(x)))
(TransformerBlock.forward, moc/model.py:31-64,83-84), as one autograd Function
over the library's kernels: the norm as a row kernel, the projections on the
MFMA engine, causal attention with RoPE inside (moc_amd/csrc/attn.hip), the
residual added in out_proj's epilogue.  The stock composition (about 45
elementwise launches a step besides the products) stays for everything else.

bf16 models and f32 models under bf16 autocast; the rounding points are the
stock ones where it stores bf16 (norm output, q/k/v, rotated q and k, the
attention output, out_proj's output), f32 in between.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn

from . import kernels as K

BF16, F32 = torch.bfloat16, torch.float32
# False: the block runs its attention half as the stock composition (the tests
# compare the two)
FUSE_BLOCK_ATTENTION = True


def stream_dtype(x):
    """The residual stream's dtype if the fused halves take it: bf16 outside
    autocast, f32 under bf16 autocast; else None."""
    if not x.is_cuda:
        return None
    if torch.is_autocast_enabled("cuda"):
        return F32 if x.dtype == F32 and torch.get_autocast_dtype("cuda") == BF16 else None
    return BF16 if x.dtype == BF16 else None


def bare(*modules) -> bool:
    """No hooks on the modules that a fused half does not call."""
    return not any(m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                   for m in modules)


def attention_half_ok(x, norm, norm_type, attn, attn_type) -> bool:
    """True if attention_half takes this block: plain modules of the model's
    own types in the stream's dtype, heads of 64 or 128, hidden up to 4096, two
    tokens or more (a gradient product over one token has no aligned operand)."""
    if not FUSE_BLOCK_ATTENTION or type(norm) is not norm_type or type(attn) is not attn_type or x.dim() != 3:
        return False
    dt = stream_dtype(x)
    qkv, out = attn.qkv_proj, attn.out_proj
    if dt is None or type(qkv) is not nn.Linear or type(out) is not nn.Linear or \
            qkv.bias is not None or out.bias is not None or not bare(norm, attn, qkv, out):
        return False
    d = x.shape[-1]
    if attn.head_dim not in (64, 128) or d != attn.num_heads * attn.head_dim or d > 4096 or x.numel() < 2 * d or \
            x.shape[1] > attn.rope_cos.shape[0] or x.shape[0] > 65535:
        return False
    return all(t.dtype == dt and t.is_contiguous() and t.device == x.device and t.data_ptr() % 16 == 0
               for t in (norm.weight, qkv.weight, out.weight, attn.rope_cos, attn.rope_sin))


def attention_half(x, norm, attn) -> torch.Tensor:
    """x + attn(norm(x)); attention_half_ok must hold."""
    return _AttentionHalf.apply(x, norm.weight, attn.qkv_proj.weight, attn.out_proj.weight, attn.rope_cos,
                                attn.rope_sin, float(norm.eps), attn.num_heads)


class _AttentionHalf(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, norm_w, qkv_w, out_w, cos, sin, eps, heads):
        batch, seq, d = x.shape
        x2 = x.reshape(-1, d).contiguous()
        scale = 1.0 / math.sqrt(d // heads)
        if x.dtype == F32:
            wq, wo = K.cast_bf16(qkv_w, out_w)
            xn, rstd = K.rmsnorm_rows_f32(x2, norm_w, eps)
        else:
            wq, wo = qkv_w, out_w
            xn, rstd = K.rmsnorm_rows(x2, norm_w, eps)
        qkv = K.linear(xn, wq)
        o, lse = K.rope_attention(qkv, batch, seq, heads, cos, sin, scale)
        if x.dtype == F32:
            h = x2 + K.linear(o, wo)
        else:
            h = K.gemm(o, wo.t(), residual=x2)
        # under autocast the casts are kept for the backward, as autocast keeps them
        ctx.save_for_backward(x2, rstd, norm_w, xn, qkv, o, lse, wq, wo, cos, sin)
        ctx.shape, ctx.heads, ctx.scale = x.shape, heads, scale
        ctx.grad_dtype = qkv_w.dtype
        return h.reshape(x.shape)

    @staticmethod
    def backward(ctx, dh):
        x2, rstd, norm_w, xn, qkv, o, lse, wq, wo, cos, sin = ctx.saved_tensors
        batch, seq, d = ctx.shape
        dh2 = dh.reshape(-1, d).contiguous()
        go = K.aligned_rows(dh2.to(BF16))
        gdt = ctx.grad_dtype
        d_out = K.gemm(go.t(), o, out_dtype=gdt)
        do = K.gemm(go, wo)
        dqkv = K.rope_attention_backward(qkv, batch, seq, ctx.heads, cos, sin, ctx.scale, o, lse, do)
        d_qkv = K.gemm(dqkv.t(), xn, out_dtype=gdt)
        dxn = K.gemm(dqkv, wq)
        if x2.dtype == F32:
            dx, dn = K.rmsnorm_backward_f32(x2, norm_w, rstd, dxn, dres=dh2)
        else:
            dx, dn = K.rmsnorm_backward(x2, norm_w, rstd, dxn, dres=go)
        return dx.reshape(ctx.shape), dn, d_qkv, d_out, None, None, None, None
