"""The attention half of a decoder block, x + out_proj(attention(norm(x)))
(TransformerBlock.forward, moc/model.py:31-64,83-84), as one autograd Function
over the library's kernels: the norm as a row kernel, the projections on the
MFMA engine, causal attention with RoPE inside (moc_amd/csrc/attn.hip), the
residual added in out_proj's epilogue.  The stock composition (about 45
elementwise launches a step besides the products) stays for everything else.
And the model's last steps: final norm with LM head, next-token loss
(moc_amd/csrc/loss.hip).

bf16 models and f32 models under bf16 autocast; the rounding points are the
stock ones where it stores bf16 (norm output, q/k/v, rotated q and k, the
attention output, out_proj's output), f32 in between.
"""
from __future__ import annotations

import math
from functools import lru_cache

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules.module import _has_any_global_hook

from . import _native as N
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


# The methods that the fused halves compute themselves.
_STOCK = {nn.Linear.forward}


def stock_method(name: str = "forward"):
    """Class decorator: a fused half may stand in for this method of the class."""
    def mark(cls):
        _STOCK.add(getattr(cls, name))
        return cls
    return mark


def runs_stock(m: nn.Module, name: str = "forward") -> bool:
    """Calling m.<name> runs a method a fused half knows: none of the
    instance's own, of a subclass's, or put in the class's place."""
    return name not in m.__dict__ and getattr(type(m), name) in _STOCK


def plain(*tensors) -> bool:
    """Tensors whose storage holds their values, which the kernels read: no
    subclass (sharded, quantised, ...) with operators of its own."""
    return all(type(t) is torch.Tensor or type(t) is nn.Parameter for t in tensors)


def bare(*modules) -> bool:
    """The modules that a fused half does not call have the forward it computes
    and no hooks, their own or those registered for every module."""
    return not _has_any_global_hook() and not any(
        m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks or not runs_stock(m)
        for m in modules)


def graph_grads(half, inputs, needs, grad):
    """The gradients of half(*inputs) with a graph of their own, for a backward
    that is to be differentiated: half is written in f32 tensor operations, which
    have derivatives of every order (autocast off), inputs are the Function's."""
    wanted = [t for t, need in zip(inputs, needs) if need]
    with torch.autocast("cuda", enabled=False):
        out = half(*inputs)
        grads = iter(torch.autograd.grad(out, wanted, grad.to(out.dtype), create_graph=True))
    return [next(grads) if need else None for need in needs]


def rms_norm_f32(x, w, eps: float):
    """x / rms(x) * w of an f32 x."""
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.float()


# Longest sequence of the fused half; from there on the stock composition over
# the library's attention is as fast or faster.  Stock time over fused, forward +
# backward, 4096 tokens a pass (the last column one sequence of 8192):
#   hidden, heads of        256    1024   4096   8192
#   bf16 1024, 64           3.72   2.37   1.17   0.98
#   bf16 1024, 128          3.50   1.98   1.18   0.78
#   bf16 2048, 64           2.14   1.67   1.03   0.96
#   bf16 2048, 128          1.99   1.56   1.00   0.76
#   f32  1024, 64           3.83   2.70   1.40   1.17
#   f32  2048, 128             -   1.71   1.12   0.84
# (forward alone 0.97 to 2.0 at 4096, 0.65 to 1.4 at 8192; one sequence of 2 to
# 2048 positions 1.3 to 8.5).
MAX_SEQ = 4096


def attention_half_ok(x, norm, norm_type, attn, attn_type) -> bool:
    """True if attention_half takes this block: plain modules of the model's
    own types in the stream's dtype, heads of 64 or 128, hidden up to 4096, up
    to MAX_SEQ positions, two tokens or more (a gradient product over one token
    has no aligned operand).  Every shape is compared: the kernels take their
    sizes from x alone."""
    if not FUSE_BLOCK_ATTENTION or type(norm) is not norm_type or type(attn) is not attn_type or x.dim() != 3:
        return False
    dt = stream_dtype(x)
    qkv, out = attn.qkv_proj, attn.out_proj
    if dt is None or type(qkv) is not nn.Linear or type(out) is not nn.Linear or \
            qkv.bias is not None or out.bias is not None or not bare(norm, attn, qkv, out):
        return False
    d = x.shape[-1]
    if attn.head_dim not in (64, 128) or d != attn.num_heads * attn.head_dim or d > 4096 or x.numel() < 2 * d or \
            x.shape[0] > 65535 or x.shape[1] > MAX_SEQ or 3 * x.numel() * 2 >= K.OPERAND_BYTES:
        return False
    cos = attn.rope_cos
    if norm.weight.shape != (d,) or qkv.weight.shape != (3 * d, d) or out.weight.shape != (d, d) or \
            cos.dim() != 2 or cos.shape[0] < x.shape[1] or cos.shape[1] != attn.head_dim // 2 or \
            attn.rope_sin.shape != cos.shape:
        return False
    read = norm.weight, qkv.weight, out.weight, attn.rope_cos, attn.rope_sin
    if not plain(x, *read) or (x.is_contiguous() and x.data_ptr() % 16):
        return False
    return all(t.dtype == dt and t.is_contiguous() and t.device == x.device and t.data_ptr() % 16 == 0 for t in read)


def attention_half(x, norm, attn) -> torch.Tensor:
    """x + attn(norm(x)); attention_half_ok must hold."""
    return _AttentionHalf.apply(x, norm.weight, attn.qkv_proj.weight, attn.out_proj.weight, attn.rope_cos,
                                attn.rope_sin, float(norm.eps), attn.num_heads)


@lru_cache(maxsize=256)
def _sizes(device_index: int, batch: int, seq: int, heads: int, head_dim: int, f32: int):
    """(saved buffer, backward scratch, GEMM workspace) bytes of a shape."""
    return (N.query("moc_attention_half_saved_size", batch, seq, heads, head_dim, f32),
            N.query("moc_attention_half_scratch_size", batch, seq, heads, head_dim, f32),
            N.query("moc_attention_half_workspace_size", batch * seq, heads * head_dim))


def _attention_f32(x, norm_w, qkv_w, out_w, cos, sin, eps: float, heads: int):
    """x + out_proj(attention(norm(x))) in f32 tensor operations."""
    b, n, d = x.shape
    q, k, v = F.linear(rms_norm_f32(x.float(), norm_w, eps), qkv_w.float()).view(b, n, 3, heads, d // heads).permute(
        2, 0, 3, 1, 4)
    c, s = cos[:n].float(), sin[:n].float()
    q, k = (torch.stack((t[..., 0::2] * c - t[..., 1::2] * s, t[..., 0::2] * s + t[..., 1::2] * c), -1).flatten(-2)
            for t in (q, k))
    later = torch.ones(n, n, dtype=torch.bool, device=x.device).triu(1)
    p = torch.softmax((q @ k.transpose(-1, -2) / math.sqrt(d // heads)).masked_fill(later, -math.inf), -1)
    return x + F.linear((p @ v).permute(0, 2, 1, 3).reshape(b, n, d), out_w.float())


class _AttentionHalf(torch.autograd.Function):
    """One native call per pass; between them one buffer of the forward's
    results (norm output, q/k/v, attention output, row factors and, under
    autocast, the weights' casts, which autocast keeps too)."""

    @staticmethod
    def forward(ctx, x, norm_w, qkv_w, out_w, cos, sin, eps, heads):
        batch, seq, d = x.shape
        given, x = x, x.contiguous()
        f32 = int(x.dtype == F32)
        dev = x.device
        nsaved, _, nws = _sizes(dev.index, batch, seq, heads, d // heads, f32)
        saved = torch.empty(nsaved, dtype=torch.uint8, device=dev)
        h = torch.empty_like(x)
        y = torch.empty((batch * seq, d), dtype=BF16, device=dev) if f32 else None
        ws = K._gemm_workspace(dev, nws) if nws > 0 else None
        scale = 1.0 / math.sqrt(d // heads)
        N.call("moc_attention_half_forward", batch, seq, heads, d // heads, f32, x.data_ptr(), norm_w.data_ptr(),
               eps, qkv_w.data_ptr(), out_w.data_ptr(), cos.data_ptr(), sin.data_ptr(), scale, h.data_ptr(),
               saved.data_ptr(), nsaved, N.ptr(y), N.ptr(ws), nws, N.stream_of(x))
        ctx.save_for_backward(given, norm_w, qkv_w, out_w, cos, sin, saved)
        ctx.heads, ctx.scale, ctx.eps = heads, scale, eps
        return h

    @staticmethod
    def backward(ctx, dh):
        x, norm_w, qkv_w, out_w, cos, sin, saved = ctx.saved_tensors
        if torch.is_grad_enabled():
            return (*graph_grads(lambda *t: _attention_f32(*t, cos, sin, ctx.eps, ctx.heads),
                                 (x, norm_w, qkv_w, out_w), ctx.needs_input_grad[:4], dh), None, None, None, None)
        x = x.contiguous()
        batch, seq, d = x.shape
        heads = ctx.heads
        f32 = int(x.dtype == F32)
        dev = x.device
        _, nscratch, nws = _sizes(dev.index, batch, seq, heads, d // heads, f32)
        dh = dh.to(x.dtype).contiguous()
        if dh.data_ptr() % 16:
            dh = dh.clone()
        scratch = torch.empty(nscratch, dtype=torch.uint8, device=dev)
        ws = K._gemm_workspace(dev, nws) if nws > 0 else None
        stream, norm, qkv, out = ctx.needs_input_grad[:4]  # dx and dn come from one kernel
        dx, dn, dq, do = (torch.empty_like(t) if need else None for t, need in (
            (x, stream or norm), (norm_w, stream or norm), (qkv_w, qkv), (out_w, out)))
        N.call("moc_attention_half_backward", batch, seq, heads, d // heads, f32, dh.data_ptr(), x.data_ptr(),
               norm_w.data_ptr(), qkv_w.data_ptr(), out_w.data_ptr(), cos.data_ptr(), sin.data_ptr(), ctx.scale,
               saved.data_ptr(), saved.numel(), N.ptr(dx), N.ptr(dn), N.ptr(dq), N.ptr(do),
               scratch.data_ptr(), nscratch, N.ptr(ws), nws, N.stream_of(x))
        return dx, dn, dq, do, None, None, None, None


def lm_head_ok(h, norm, norm_type, head, weight) -> bool:
    """True if lm_head takes the model's last step, weight @ norm(h): plain
    modules (head: the nn.Linear that holds weight, or None for a tied one) in
    the stream's dtype, two tokens or more."""
    dt = stream_dtype(h)
    if dt is None or type(norm) is not norm_type or h.dim() != 3 or not bare(norm):
        return False
    if head is not None and (type(head) is not nn.Linear or head.bias is not None or not bare(head)):
        return False
    d = h.shape[-1]
    if not plain(h, norm.weight, weight) or d % 8 or d > 4096 or weight.dim() != 2 or weight.shape[0] % 8 or \
            h.numel() < 2 * d:
        return False
    return all(t.dtype == dt and t.is_contiguous() and t.device == h.device and t.data_ptr() % 16 == 0
               for t in (h, norm.weight, weight)) and norm.weight.shape == (d,) and weight.shape[1] == d


def lm_head(h, norm, weight) -> torch.Tensor:
    """norm(h) @ weight.T as bf16 logits; lm_head_ok must hold."""
    return _LMHead.apply(h, norm.weight, weight, float(norm.eps))


def _own_head_dx(tokens: int, d: int, vocab: int) -> bool:
    """dX contracts over the vocabulary into few tiles: the library's product
    leaves most CUs idle, the engine's splits K.  Library and engine, us, of 32000
    words: 93 / 44 (16 tokens, d 512), 104 / 32 (512, 512), 289 / 127 (4096,
    512), 325 / 227 (4096, 1024), 427 / 406 (4096, 2048), the last of the range
    where the engine was ahead.  1000 to 128256 words: the engine at most 4 %
    behind anywhere in it (8192 words, d 1024, 8192 tokens: 117 / 121)."""
    return tokens * d <= 1 << 23 and 2 * vocab * max(tokens, d) < K.OPERAND_BYTES


def _own_head_dw(d: int, vocab: int, tokens: int) -> bool:
    """dW on the engine where its 256-wide tiles fill their rounds of 256 CUs:
    0.8 of one round, 0.7 of several.  Library and engine, us, 4096 tokens: 131 /
    108 (32000 words, d 512: 250 tiles), 109 / 108 (26624: 208), 249 / 210 (32000,
    d 1024: 500), 178 / 171 (16384, d 1536: 384); but 68 / 75 (16384, d 512: 128;
    23 / 37 at 1024 tokens), 90 / 98 (24576: 192), 124 / 169 (24576, d 640: 288).
    Narrower or with fewer words the engine is ahead or behind by the token count
    (32000 words, d 256, 512 tokens 20 / 18; 8192, d 1024, 8192 tokens 137 / 123)
    and the library keeps them."""
    tiles = -(-d // 256) * -(-vocab // 256)
    rounds = -(-tiles // 256)
    return (d >= 512 and vocab >= 16384 and tiles >= (0.8 if rounds == 1 else 0.7) * 256 * rounds
            and 2 * tokens * max(vocab, d) < K.OPERAND_BYTES)


class _LMHead(torch.autograd.Function):
    """The final norm as one row kernel each way (f32 stream: straight to the
    product's bf16 operand), the forward product by the library (equal to the
    engine's at d <= 1024: 160 and 153 us at 4096 x 512 x 32000, ahead above:
    377 and 434 at d 2048), the backward's by shape."""

    @staticmethod
    def forward(ctx, h, norm_w, weight, eps):
        d = h.shape[-1]
        h2 = h.reshape(-1, d)
        if h.dtype == F32:
            xn, rstd = K.rmsnorm_rows_f32(h2, norm_w, eps)
            wb, = K.cast_bf16(weight)
        else:
            (xn, rstd), wb = K.rmsnorm_rows(h2, norm_w, eps), weight
        ctx.save_for_backward(h, norm_w, weight, xn, rstd, wb)
        ctx.eps = eps
        return K.unaliased(torch.matmul(xn, wb.t()), (*h.shape[:-1], weight.shape[0]))

    @staticmethod
    def backward(ctx, g):
        h, norm_w, weight, xn, rstd, wb = ctx.saved_tensors
        if torch.is_grad_enabled():  # a graph of the gradient is wanted: the stock operators have one
            xf = h.float()
            y = (xf * torch.rsqrt(torch.mean(xf * xf, dim=-1, keepdim=True) + ctx.eps)).to(h.dtype) * norm_w
            wanted = [t for t in (h, norm_w, weight) if t.requires_grad]
            it = iter(torch.autograd.grad(y.to(BF16) @ weight.to(BF16).t(), wanted, g, create_graph=True))
            return (*(next(it) if t.requires_grad else None for t in (h, norm_w, weight)), None)
        d, vocab = h.shape[-1], weight.shape[0]
        # contiguous: an expanded gradient has rows 0 apart, which no GEMM operand has
        h2, g2 = h.reshape(-1, d), g.contiguous().reshape(-1, vocab)
        dh = dnw = dw = None
        if ctx.needs_input_grad[0] or ctx.needs_input_grad[1]:
            dxn = K.gemm(g2, wb) if _own_head_dx(h2.shape[0], d, vocab) else torch.matmul(g2, wb)
            dh, dnw = (K.rmsnorm_backward_f32 if h.dtype == F32 else K.rmsnorm_backward)(h2, norm_w, rstd, dxn)
            dh = dh.reshape(h.shape)
        if ctx.needs_input_grad[2]:
            dw = (K.gemm(g2.t(), xn, out_dtype=weight.dtype) if _own_head_dw(d, vocab, h2.shape[0])
                  else torch.matmul(g2.t(), xn).to(weight.dtype))
        return dh, dnw, dw, None


def next_token_loss_ok(logits, labels) -> bool:
    """True if next_token_loss takes these: bf16 device logits whose stock loss
    is f32 (autocast) or bf16, int64 labels of their shape."""
    return (plain(logits, labels) and logits.is_cuda and logits.dtype == BF16 and logits.dim() == 3
            and logits.shape[1] >= 2
            and logits.is_contiguous() and logits.data_ptr() % 16 == 0 and logits.numel() > 0
            and logits.shape[2] % 8 == 0 and logits.shape[2] <= 65536 and logits.shape[0] * logits.shape[1] <= 1 << 22
            and labels.device == logits.device and labels.dtype == torch.int64
            and labels.shape == logits.shape[:2])


def next_token_loss(logits, labels, ignore_index: int = -100) -> torch.Tensor:
    """F.cross_entropy(logits[:, :-1], labels[:, 1:], ignore_index) of bf16
    logits, f32 under autocast (as autocast runs it), else bf16;
    next_token_loss_ok must hold."""
    f32 = torch.is_autocast_enabled("cuda")
    return _NextTokenLoss.apply(logits, labels.contiguous(), ignore_index, F32 if f32 else BF16)[0]


class _NextTokenLoss(torch.autograd.Function):
    """(loss, the logits as it saw them, which nobody else holds): the backward
    reads the second, so a caller may write its logits in place before it."""

    @staticmethod
    def forward(ctx, logits, labels, ignore_index, dtype):
        b, s, v = logits.shape
        buf = torch.empty(2 * b * s + 1, dtype=F32, device=logits.device)  # lse, row losses, 1 / count
        loss = torch.empty((), dtype=dtype, device=logits.device)
        seen = torch.empty_like(logits) if ctx.needs_input_grad[0] else None
        p = buf.data_ptr()
        N.call("moc_next_token_loss_forward_keep", logits.data_ptr(), v, b, s, v, labels.data_ptr(), ignore_index, p,
               p + 4 * b * s, loss.data_ptr(), N.dtype_code(dtype), p + 8 * b * s, N.ptr(seen), v,
               N.stream_of(logits))
        ctx.save_for_backward(seen, labels, buf)
        ctx.ignore_index = ignore_index
        ctx.set_materialize_grads(False)
        return loss, seen

    @staticmethod
    def backward(ctx, g, g_seen):
        if g is None:  # the second pass of a second derivative: d seen / d logits
            return g_seen, None, None, None
        seen, labels, buf = ctx.saved_tensors
        if torch.is_grad_enabled():  # a graph of the gradient is wanted: the stock loss has one
            x = seen[:, :-1].flatten(0, 1)
            loss = F.cross_entropy(x.float() if g.dtype == F32 else x, labels[:, 1:].flatten(),
                                   ignore_index=ctx.ignore_index)
            d = torch.autograd.grad(loss, seen, g, create_graph=True)[0]
        else:
            b, s, v = seen.shape
            d = torch.empty_like(seen)
            g = g.contiguous()
            p = buf.data_ptr()
            N.call("moc_next_token_loss_backward", seen.data_ptr(), v, b, s, v, labels.data_ptr(), ctx.ignore_index,
                   p, p + 8 * b * s, g.data_ptr(), N.dtype_code(g.dtype), d.data_ptr(), v, N.stream_of(seen))
        return d if g_seen is None else d + g_seen, None, None, None
