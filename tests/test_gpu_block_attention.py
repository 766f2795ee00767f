"""The decoder block's fused attention half and its kernels (causal attention
with RoPE, the f32-stream norm, the multi-matrix cast) against 64 bits and the
stock composition."""
import math

import pytest
import torch

import moc_amd.block as B
from moc_amd import MoCConfig, build_ffn
from moc_amd import kernels as K
from moc_amd.model import CausalSelfAttention, RMSNorm, TransformerBlock, rotary_tables, rotate_pairs

pytestmark = pytest.mark.gpu
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64


def _rot(x, c, s):
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)


@pytest.mark.parametrize("seq", [1, 2, 31, 33, 64, 65, 127, 129, 200, 256, 300, 513])
@pytest.mark.parametrize("heads,dim,table", [(3, 64, BF), (2, 64, F32), (2, 128, BF)])
def test_rope_attention(seq, heads, dim, table):
    batch = 2
    g = torch.Generator(device="cuda").manual_seed(seq * heads + dim)
    t, d = batch * seq, heads * dim
    qkv = torch.randn(t, 3 * d, generator=g, device="cuda").to(BF)
    go = torch.randn(t, d, generator=g, device="cuda").to(BF)
    cos, sin = (x.to("cuda", table) for x in rotary_tables(dim, seq + 3))
    scale = 1.0 / math.sqrt(dim)
    o, lse = K.rope_attention(qkv, batch, seq, heads, cos, sin, scale)
    dqkv = K.rope_attention_backward(qkv, batch, seq, heads, cos, sin, scale, o, lse, go)
    assert all(torch.equal(a, b) for a, b in zip((o, lse), K.rope_attention(qkv, batch, seq, heads, cos, sin, scale)))

    c, s = cos[:seq].to(F64), sin[:seq].to(F64)
    q, k, v = qkv.to(F64).view(batch, seq, 3, heads, dim).permute(2, 0, 3, 1, 4)
    if table == BF:  # bf16 tensor operations: each product and the sum rounded
        q, k = (_rot(x.to(BF), cos[:seq], sin[:seq]).to(F64) for x in (q, k))
    else:
        q, k = (_rot(x.float(), cos[:seq], sin[:seq]).to(BF).to(F64) for x in (q, k))
    gg = go.to(F64).view(batch, seq, heads, dim).transpose(1, 2)
    sc = (q @ k.transpose(-1, -2)) * scale + torch.full((seq, seq), -math.inf, device="cuda", dtype=F64).triu(1)
    p = torch.softmax(sc, -1)
    ref = p @ v
    # o: its rounding, and P's to bf16 in the product
    e8 = 2.0 ** -8
    ob = o.to(F64).view(batch, seq, heads, dim).transpose(1, 2)
    assert ((ob - ref).abs() <= e8 * (ref.abs() + 2 * p @ v.abs()) + 1e-5).all()
    want = torch.logsumexp(sc, -1) / math.log(2.0)
    assert ((lse.to(F64) - want).abs() <= 1e-5 * (1 + want.abs())).all()
    # dS = P (dP - delta) scale; delta comes from the rounded o, dS is rounded
    dp = gg @ v.transpose(-1, -2)
    delta = (gg * ref).sum(-1, keepdim=True)
    ds = p * (dp - delta)
    ds_err = p * (e8 * (gg.abs() * (ref.abs() + 2 * p @ v.abs())).sum(-1, keepdim=True)) + 2 * e8 * ds.abs()
    grads = {"q": (ds @ k * scale, ds_err @ k.abs() * scale),
             "k": (ds.transpose(-1, -2) @ q * scale, ds_err.transpose(-1, -2) @ q.abs() * scale),
             "v": (p.transpose(-1, -2) @ gg, 2 * e8 * p.transpose(-1, -2) @ gg.abs())}
    got = dict(zip("qkv", dqkv.to(F64).view(batch, seq, 3, heads, dim).permute(2, 0, 3, 1, 4)))
    for n, (r, err) in grads.items():
        if n != "v":  # rotated back: each value mixes its pair
            r = _rot(r, c, -s)
            err = (err[..., 0::2] + err[..., 1::2]).repeat_interleave(2, -1)
        bad = (got[n] - r).abs() > e8 * r.abs() + err + 1e-5
        assert not bad.any(), (n, int(bad.sum()))


def _pair(dtype, hidden, heads, seq, seed):
    torch.manual_seed(seed)
    cfg = MoCConfig(hidden_size=hidden, intermediate_size=2 * hidden, num_hidden_layers=1,
                    num_attention_heads=heads, vocab_size=32, max_seq_len=max(seq, 8))
    norm, attn = RMSNorm(hidden), CausalSelfAttention(cfg)
    norm.weight.data += 0.1 * torch.randn(hidden)
    return norm.to("cuda", dtype), attn.to("cuda", dtype)


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("batch,seq,hidden,heads", [(2, 1, 64, 1), (3, 77, 256, 4), (2, 256, 512, 8),
                                                    (1, 130, 256, 2)])
def test_attention_half_matches_the_stock_composition(dtype, batch, seq, hidden, heads):
    norm, attn = _pair(dtype, hidden, heads, seq, 7)
    ref_n, ref_a = _pair(F64, hidden, heads, seq, 7)
    for m, r in ((norm, ref_n), (attn, ref_a)):
        for a, b in zip(m.parameters(), r.parameters()):
            b.data.copy_(a.data)
    x = torch.randn(batch, seq, hidden, device="cuda").to(dtype)
    dh = torch.randn(batch, seq, hidden, device="cuda").to(dtype)

    def run(fn, n, a, xx, gg, cast):
        xx = xx.clone().requires_grad_()
        with torch.autocast("cuda", dtype=BF, enabled=cast):
            if fn is B.attention_half:
                assert B.attention_half_ok(xx, n, RMSNorm, a, CausalSelfAttention)
            y = fn(xx, n, a)
        grads = torch.autograd.grad(y, [xx, n.weight, a.qkv_proj.weight, a.out_proj.weight], gg)
        return [y - xx, *grads]

    stock = lambda xx, n, a: xx + a(n(xx))  # noqa: E731
    cast = dtype == F32
    got = run(B.attention_half, norm, attn, x, dh, cast)
    old = run(stock, norm, attn, x, dh, cast)
    exact = run(stock, ref_n, ref_a, x.to(F64), dh.to(F64), False)
    for g, o, e in zip(got, old, exact):
        assert g.dtype == o.dtype and g.shape == o.shape
        err = lambda t: ((t.to(F64) - e).norm() / e.norm().clamp_min(1e-12)).item()  # noqa: E731
        # no further from 64 bits than the stock composition
        assert err(g) <= 1.1 * err(o) + 1e-4, (err(g), err(o))


def test_block_takes_the_fused_half_and_hooks_keep_the_stock_one():
    cfg = MoCConfig(hidden_size=256, intermediate_size=512, num_hidden_layers=1, num_attention_heads=4, vocab_size=32)
    blk = TransformerBlock(cfg, "moc").to("cuda", BF)
    x = torch.randn(2, 40, 256, device="cuda").to(BF)
    calls = []
    blk.attn.register_forward_hook(lambda *a: calls.append(1))
    y1 = blk(x)
    assert calls
    blk.attn._forward_hooks.clear()
    y2 = blk(x)
    assert len(calls) == 1
    assert (y1.float() - y2.float()).norm() <= 2e-2 * y1.float().norm()
    from torch.utils.checkpoint import checkpoint
    xs = [x.clone().requires_grad_() for _ in range(2)]
    blk(xs[0]).sum().backward()
    g0 = [p.grad.clone() for p in blk.parameters()]
    blk.zero_grad()
    checkpoint(blk, xs[1], use_reentrant=False).sum().backward()
    assert torch.equal(xs[0].grad, xs[1].grad)
    assert all(torch.equal(a, p.grad) for a, p in zip(g0, blk.parameters()))


@pytest.mark.parametrize("rows,d", [(1, 8), (5, 64), (37, 520), (300, 1024), (9, 4096)])
def test_rmsnorm_f32(rows, d):
    g = torch.Generator(device="cuda").manual_seed(rows + d)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, w, dres, dy = r(rows, d), 1 + 0.1 * r(d), r(rows, d), r(rows, d).to(BF)
    y, rstd = K.rmsnorm_rows_f32(x, w, 1e-6)
    xd, wd = x.to(F64).requires_grad_(), w.to(F64).requires_grad_()
    ref = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-6) * wd
    assert ((y.to(F64) - ref).abs() <= (2.0 ** -8 + 1e-5) * ref.abs()).all()
    dx, dw = K.rmsnorm_backward_f32(x, w, rstd, dy, dres)
    gx, gw = torch.autograd.grad(ref, [xd, wd], dy.to(F64))
    gx = gx + dres.to(F64)
    n = xd.detach() * rstd.to(F64)[:, None]
    # f32 sums: d (rows) terms of the products' magnitudes
    mag = dres.abs().to(F64) + (dy.to(F64) * wd * rstd.to(F64)[:, None]).abs() * (1 + n.abs())
    assert ((dx.to(F64) - gx).abs() <= 1e-6 * (d ** 0.5) * mag + 1e-6).all()
    assert ((dw.to(F64) - gw).abs() <= 1e-5 * (dy.to(F64) * n).abs().sum(0) + 1e-6).all()


def test_cast_bf16():
    g = torch.Generator(device="cuda").manual_seed(3)
    mats = [torch.randn(r, c, generator=g, device="cuda") for r, c in
            ((1, 1), (3, 7), (64, 64), (5, 1001), (2048, 5461), (33, 8), (10, 12), (7, 4), (128, 100), (2, 3))]
    mats[2][0, :4] = torch.tensor([float("nan"), float("inf"), -float("inf"), -0.0])
    for m, c in zip(mats, K.cast_bf16(*mats)):
        assert c.stride(0) % 8 == 0 and c.data_ptr() % 16 == 0
        assert torch.equal(c.contiguous().view(torch.int16), m.to(BF).view(torch.int16))


@pytest.mark.parametrize("ffn_type", ["moc", "moc_gcp", "moc_2_8", "moc_post_silu_abs"])
@pytest.mark.parametrize("inter", [320, 333])
def test_ffn_half_under_autocast_matches_the_stock_composition(ffn_type, inter):
    """h + ffn(norm(h)) of an f32 block under autocast: the norm's output, so
    the FFN's bf16 input, is the stock one but for f32 sums in another order."""
    import moc_amd.ffn as FF
    torch.manual_seed(3)
    cfg = MoCConfig(hidden_size=128, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=2, vocab_size=32)
    blk = TransformerBlock(cfg, ffn_type).to("cuda")
    h = torch.randn(3, 50, 128, device="cuda")
    dy = torch.randn_like(h)

    def run(fused):
        x = h.clone().requires_grad_()
        with torch.autocast("cuda", dtype=BF):
            if fused:
                assert FF.block_ffn_f32_ok(x, blk.ffn_norm.weight, blk.ffn)
                y = FF.block_ffn(x, blk.ffn_norm.weight, blk.ffn_norm.eps, blk.ffn)
            else:
                y = x + blk.ffn(blk.ffn_norm(x))
        ps = [blk.ffn_norm.weight, *blk.ffn.parameters()]
        return [y - x, *torch.autograd.grad(y, [x, *ps], dy)]

    for a, b in zip(run(True), run(False)):
        assert a.dtype == b.dtype == F32 and a.shape == b.shape
        assert (a - b).norm() <= 5e-3 * b.norm()


@pytest.mark.parametrize("mode", ["moc", "moc_gcp", "moc_2_8", "moc_post_silu_abs"])
@pytest.mark.parametrize("dtype,tokens", [(F32, 2), (F32, 300), ("autocast", 2), ("autocast", 300)])
def test_one_call_passes_equal_the_separate_launches(mode, dtype, tokens):
    """The one-call f32 layer and the one-call f32-stream FFN half against the
    same launches issued one by one: bit for bit."""
    import moc_amd.ffn as FF
    torch.manual_seed(tokens)
    cfg = MoCConfig(hidden_size=128, intermediate_size=344, num_hidden_layers=1, num_attention_heads=2, vocab_size=32)
    blk = TransformerBlock(cfg, mode).to("cuda")
    h = torch.randn(tokens, 128, device="cuda")

    def run(native):
        FF.USE_NATIVE_LAYER = native
        try:
            x = h.clone().requires_grad_()
            with torch.autocast("cuda", dtype=BF, enabled=dtype == "autocast"):
                y = FF.block_ffn(x, blk.ffn_norm.weight, 1e-6, blk.ffn) if dtype == "autocast" else blk.ffn(x)
            ps = list(blk.ffn.parameters()) + ([blk.ffn_norm.weight] if dtype == "autocast" else [])
            return [y, *torch.autograd.grad(y, [x, *ps], h.sin())]
        finally:
            FF.USE_NATIVE_LAYER = True

    for a, b in zip(run(True), run(False)):
        # the bf16 passes group the weight gradients' split-K sums differently
        if dtype == "autocast" and tokens > 2:
            assert (a - b).norm() <= 1e-5 * b.norm() + (2e-3 * b.norm() if a.shape == h.shape else 0)
        else:
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,tokens,inter", [(BF, 80, 512), (F32, 80, 512), (F32, 80, 333), (BF, 80, 333),
                                                (BF, 2, 512), (F32, 2, 512)])
def test_block_output_takes_writes_in_place(dtype, tokens, inter):
    """A forward hook that adds to the stream in place, as h + ffn(norm(h)) allows."""
    torch.manual_seed(5)
    cfg = MoCConfig(hidden_size=256, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=4,
                    vocab_size=32)
    blk = TransformerBlock(cfg, "moc").to("cuda", dtype)
    x = torch.randn(1, tokens, 256, device="cuda").to(dtype).requires_grad_()
    with torch.autocast("cuda", dtype=BF, enabled=dtype == F32):
        want = blk(x)
        hook = blk.register_forward_hook(lambda m, a, y: y.add_(1.0))
        got = blk(x)
        hook.remove()
    assert torch.equal(got, want + 1)
    assert all(torch.equal(*g) for g in zip(*(torch.autograd.grad(y, [x, *blk.parameters()], y.detach().sign())
                                              for y in (got, want + 1))))


@pytest.mark.parametrize("dtype", [BF, F32])
def test_ffn_output_takes_writes_in_place(dtype):
    ffn = build_ffn(256, 512, "moc", k=128).to("cuda", dtype)
    x = torch.randn(2, 40, 256, device="cuda").to(dtype).requires_grad_()
    want = ffn(x)
    got = ffn(x)
    got.mul_(2.0)
    assert torch.equal(got, 2 * want)
    assert torch.equal(torch.autograd.grad(got.sum(), x)[0], torch.autograd.grad((2 * want).sum(), x)[0])


@pytest.mark.parametrize("dtype", [BF, F32])
@pytest.mark.parametrize("wanted", [("x",), ("qkv",), ("out",), ("norm",), ("x", "out"), ("norm", "qkv"), ("qkv", "out"),
                                    ("x", "norm", "qkv", "out")])
def test_attention_half_leaves_frozen_operands_out(dtype, wanted):
    """Only what needs a gradient gets one, the same bits as with all of them,
    and the products of the others are not computed."""
    norm, attn = _pair(dtype, 256, 4, 40, 3)
    x = torch.randn(2, 40, 256, device="cuda").to(dtype).requires_grad_()
    dh = torch.randn(2, 40, 256, device="cuda").to(dtype)
    leaf = {"x": x, "norm": norm.weight, "qkv": attn.qkv_proj.weight, "out": attn.out_proj.weight}

    def grads(names):
        for n, t in leaf.items():
            t.requires_grad_(n in names)
        with torch.autocast("cuda", dtype=BF, enabled=dtype == F32):
            y = B.attention_half(x, norm, attn)
        seen, call = [], B.N.call
        B.N.call = lambda name, *a: seen.append((name, a)) or call(name, *a)
        try:
            return dict(zip(names, torch.autograd.grad(y, [leaf[n] for n in names], dh))), seen[-1]
        finally:
            B.N.call = call

    every, _ = grads(tuple(leaf))
    some, (name, args) = grads(wanted)
    assert name == "moc_attention_half_backward"
    assert all(torch.equal(some[n], every[n]) for n in wanted)
    dx, dn, dq, do = args[15:19]
    assert ("qkv" in wanted) == (dq is not None) and ("out" in wanted) == (do is not None)
    assert (dx is None) == (dn is None) == (not {"x", "norm"} & set(wanted))


def _dense_block64(x, blk, heads):
    """The block in 64 bits with every channel selected."""
    def norm(t, m):
        return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + m.eps) * p[m.weight]

    p = {q: q.detach().to(F64).requires_grad_() for q in blk.parameters()}
    a, f = blk.attn, blk.ffn
    n, d = x.shape[1:]
    q, k, v = (norm(x, blk.attn_norm) @ p[a.qkv_proj.weight].t()).view(-1, n, 3, heads, d // heads).permute(2, 0, 3, 1, 4)
    c, s = a.rope_cos[:n].to(F64), a.rope_sin[:n].to(F64)
    q, k = _rot(q, c, s), _rot(k, c, s)
    sc = q @ k.transpose(-1, -2) / math.sqrt(d // heads) + torch.full((n, n), -math.inf, device="cuda", dtype=F64).triu(1)
    h = x + (torch.softmax(sc, -1) @ v).permute(0, 2, 1, 3).reshape(x.shape) @ p[a.out_proj.weight].t()
    t = norm(h, blk.ffn_norm)
    g, u, w = (p[m.weight] for m in (f.gate_proj, f.up_proj, f.down_proj))
    return h + (torch.nn.functional.silu(t @ g.t()) * (t @ u.t())) @ w.t(), list(p.values())


@pytest.mark.parametrize("mode", ["moc", "moc_gcp"])
@pytest.mark.parametrize("dtype,seq,inter", [(BF, 20, 344), (F32, 20, 344), (BF, 20, 333), (F32, 20, 333)])
def test_block_second_derivative(mode, dtype, seq, inter):
    """A gradient penalty through a whole block, every channel selected so that
    rounding moves no selection, against 64 bits."""
    torch.manual_seed(6)
    cfg = MoCConfig(hidden_size=128, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=2,
                    vocab_size=32, k=inter)
    blk = TransformerBlock(cfg, mode).to("cuda", dtype)
    x = torch.randn(2, seq, 128, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(2, seq, 128, device="cuda").to(dtype)

    def penalty(y, xx, ps, dd):
        gx, = torch.autograd.grad(y, xx, dd, create_graph=True)
        return torch.autograd.grad(gx.to(F64).square().sum(), [xx, *ps])

    with torch.autocast("cuda", dtype=BF, enabled=dtype == F32):
        y = blk(x)
    got = penalty(y, x, list(blk.parameters()), dy)
    xd = x.detach().to(F64).requires_grad_()
    yd, ps = _dense_block64(xd, blk, 2)
    want = penalty(yd, xd, ps, dy.to(F64))
    for a, b, q in zip(got, want, [x, *blk.parameters()]):
        assert a.dtype == q.dtype
        # operands and stream of bf16 (2^-9 each): the forward's values, the
        # stream between the halves and, for a bf16 block, each cotangent that
        # passes it are rounded once or twice
        assert (a.to(F64) - b).norm() <= 8 * 2.0 ** -9 * b.norm(), ((a.to(F64) - b).norm() / b.norm()).item()


@pytest.mark.parametrize("mode", ["moc", "moc_2_8", "moc_post_silu_abs"])
def test_block_second_derivative_of_a_selection(mode):
    """Selected channels only: zero where no token selects a channel."""
    torch.manual_seed(7)
    cfg = MoCConfig(hidden_size=128, intermediate_size=344, num_hidden_layers=1, num_attention_heads=2,
                    vocab_size=32, k=3)
    blk = TransformerBlock(cfg, mode).to("cuda", BF)
    x = torch.randn(1, 2, 128, device="cuda").to(BF).requires_grad_()
    y = blk(x)
    to = [x, blk.ffn.gate_proj.weight, *blk.parameters()]
    first = torch.autograd.grad(y, to, torch.ones_like(y), create_graph=True)
    plain = torch.autograd.grad(blk(x), to, torch.ones_like(y))
    for a, b in zip(first, plain):
        assert a.grad_fn is not None and (a.float() - b.float()).norm() <= 2e-2 * b.float().norm()
    unused = (plain[1] == 0).all(1)
    dg, = torch.autograd.grad(first[0].float().square().sum(), blk.ffn.gate_proj.weight)
    assert dg.abs().max() > 0
    if mode != "moc_2_8":
        assert unused.any() and (dg[unused] == 0).all()


@pytest.mark.parametrize("seq", [17, 64, 128, 129, 200, 256, 257, 512, 1024])
@pytest.mark.parametrize("dim,table", [(64, BF), (64, F32), (128, BF), (128, F32)])
def test_rope_attention_rounds_where_the_library_attention_does(seq, dim, table):
    """Key tiles below, inside and above the range of the 128-key ones: few
    outputs differ from the library's (another tile size: 5 to 20 %)."""
    heads, batch = 256 // dim, 1 + 1024 // seq
    g = torch.Generator(device="cuda").manual_seed(seq)
    qkv = torch.randn(batch * seq, 3 * heads * dim, generator=g, device="cuda").to(BF)
    cos, sin = (x.to("cuda", table) for x in rotary_tables(dim, seq))
    o, _ = K.rope_attention(qkv, batch, seq, heads, cos, sin, 1 / math.sqrt(dim))
    q, k, v = qkv.view(batch, seq, 3, heads, dim).permute(2, 0, 3, 1, 4)
    q, k = (rotate_pairs(t, cos, sin).to(BF) for t in (q, k))
    r = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True)
    assert (o != r.permute(0, 2, 1, 3).reshape(o.shape)).float().mean() <= 5e-3


@pytest.mark.parametrize("dtype,inter", [(BF, 512), (F32, 512), (F32, 333)])
def test_block_takes_a_gradient_off_the_16_byte_grid(dtype, inter):
    """The gradient of a concatenation is a view into it: that of an aligned copy."""
    torch.manual_seed(9)
    cfg = MoCConfig(hidden_size=128, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=2,
                    vocab_size=32)
    blk = TransformerBlock(cfg, "moc").to("cuda", dtype)
    x = torch.randn(2, 20, 128, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(2, 20, 128, device="cuda").to(dtype)
    off = torch.cat((dy.new_zeros(1), dy.flatten()))[1:].view(dy.shape)
    assert off.data_ptr() % 16 and off.is_contiguous()
    with torch.autocast("cuda", dtype=BF, enabled=dtype == F32):
        y = blk(x)
    want = torch.autograd.grad(y, [x, *blk.parameters()], dy, retain_graph=True)
    got = torch.autograd.grad(y, [x, *blk.parameters()], off)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
