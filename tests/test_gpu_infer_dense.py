"""The dense many-token inference layer (K.ffn_infer and the module routes that
take it) against 64-bit arithmetic on inputs whose gate scores are exact."""
import pytest
import torch
import torch.nn.functional as F

from moc_amd import kernels as K
from moc_amd.inference.inference_ffn import InferenceMoCSwiGLUFFN

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _case(nb, hidden, inter, seed):
    """x in {-1, 0, 1}, weights in {-2 .. 2} / 128: every gate and up sum is
    exact in f32 and in bf16, so the selection has one right answer."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ri = lambda lo, hi, s: torch.randint(lo, hi + 1, s, generator=gen, device="cuda")  # noqa: E731
    x = ri(-1, 1, (nb, hidden)).to(BF)
    w = [(ri(-2, 2, s).float() / 128).to(BF) for s in ((inter, hidden), (inter, hidden), (hidden, inter))]
    return x, w


def _reference(x, w, k, grouped):
    wg, wu, wd = (t.double() for t in w)
    g, u = x.double() @ wg.t(), x.double() @ wu.t()
    nb, inter = g.shape
    if grouped:
        order = torch.sort(g.reshape(nb, -1, 8), dim=-1, descending=True, stable=True).indices[..., :2]
        mask = torch.zeros(nb, inter // 8, 8, device=g.device).scatter_(-1, order, 1.0).reshape(nb, inter)
        z = (F.silu(g) * u).to(BF).double()  # rounded once
    else:
        order = torch.sort(g, dim=-1, descending=True, stable=True).indices[:, :k]
        mask = torch.zeros_like(g).scatter_(-1, order, 1.0)
        z = (F.silu(g).to(BF).double() * u).to(BF).double()
    z = z * mask
    return z @ wd.t(), z.abs() @ wd.abs().t()


def _check(y, ref, mags, inter, extra=0.0):
    # one bf16 rounding of y; z may round the other way where f32 SiLU differs
    # from the 64-bit one (half an ulp of z at most, on few channels)
    bound = 2.0 ** -8 * (ref.abs() + extra) + (2.0 ** -9 + inter * 2.0 ** -24) * mags + 1e-30
    assert ((y.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("nb,hidden,inter,k", [(17, 64, 200, 1), (64, 128, 333, 100), (65, 256, 1000, 1000),
                                               (200, 512, 1376, 256), (300, 192, 5461, 1024)])
@pytest.mark.parametrize("residual", [False, True])
def test_global(nb, hidden, inter, k, residual):
    x, w = _case(nb, hidden, inter, nb + inter)
    wdt = K.down_weight_t_for_decode(w[2])
    ref, mags = _reference(x, w, k, False)
    res = torch.randn(nb, hidden, device="cuda").to(BF) if residual else None
    assert K.ffn_infer_fits(x, w[0], w[1], wdt)
    y = K.ffn_infer(x, w[0], w[1], wdt, k, residual=res)
    if residual:
        _check(y, ref + res.double(), mags, inter, extra=ref.abs())
    else:
        _check(y, ref, mags, inter)
        m = InferenceMoCSwiGLUFFN(hidden, inter, k).to("cuda", BF)
        for p, t in zip((m.gate_proj, m.up_proj, m.down_proj), w):
            p.weight.data.copy_(t)
        assert torch.equal(m(x), y)
        # the gate-given operator: the same steps from the gate scores
        g = K.linear(x, w[0])
        _check(K.global_after_gate(x, g, w[1], wdt, k), ref, mags, inter)


@pytest.mark.parametrize("nb,hidden,inter", [(17, 64, 8), (33, 128, 200), (64, 256, 1000), (513, 64, 1376),
                                             (200, 512, 2736)])
def test_28(nb, hidden, inter):
    x, w = _case(nb, hidden, inter, nb + inter)
    wdt = K.down_weight_t_for_decode(w[2])
    ref, mags = _reference(x, w, 0, True)
    y = K.ffn_infer(x, w[0], w[1], wdt, 0, grouped=True)
    _check(y, ref, mags, inter)
    m = InferenceMoCSwiGLUFFN(hidden, inter, inter // 4, grouped_a=2, grouped_b=8).to("cuda", BF)
    for p, t in zip((m.gate_proj, m.up_proj, m.down_proj), w):
        p.weight.data.copy_(t)
    assert torch.equal(m(x), y)
    run = m.make_moc2_8_graph_runner(nb)
    for s in range(3):  # replays with eager work between them
        xs = x.roll(s, 0).contiguous()
        got = run(xs).clone()
        assert torch.equal(got, m(xs))


def test_28_nan_rows_and_ties():
    """NaN gates rank first and equal ones go to the lower channel, as in the
    packed path; other tokens' rows are untouched by a NaN token."""
    x, w = _case(20, 64, 64, 1)
    x[3] = float("nan")
    x[5] = 0  # all gates equal: channels 0 and 1 of each group
    wdt = K.down_weight_t_for_decode(w[2])
    y = K.ffn_infer(x, w[0], w[1], wdt, 0, grouped=True)
    assert torch.isnan(y[3]).all() and (y[5] == 0).all()
    ref, mags = _reference(torch.nan_to_num(x), w, 0, True)
    keep = [i for i in range(20) if i != 3]
    _check(y[keep], ref[keep], mags[keep], 64)


@pytest.mark.parametrize("nb", [5, 8, 9, 16, 17, 40])
@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("hidden,inter", [(256, 704), (1024, 2736), (2048, 5464)])
def test_layer_with_norm_and_residual(nb, grouped, hidden, inter):
    """x + FFN(RMSNorm(x)) equals the layer on the row kernel's norm, plus x,
    bit for bit: the same launches with the residual in the last one."""
    gen = torch.Generator(device="cuda").manual_seed(nb + hidden)
    kw = dict(grouped_a=2, grouped_b=8) if grouped else {}
    m = InferenceMoCSwiGLUFFN(hidden, inter, inter // 4 if grouped else hidden // 2, **kw).to("cuda", BF)
    x = torch.randn(nb, hidden, generator=gen, device="cuda").to(BF)
    w = (1 + 0.1 * torch.randn(hidden, generator=gen, device="cuda")).to(BF)
    xn, _ = K.rmsnorm_rows(x, w, 1e-6)
    xf = x.float()
    stock = (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)).to(BF) * w
    # the factor's f32 sum runs in another order: an ulp of f32 decides a
    # bf16 rounding at most here and there
    assert ((xn.float() - stock.float()).abs() <= 2.0 ** -7 * stock.float().abs()).all()
    with torch.no_grad():
        y = m.fused_decode_residual(x, w, 1e-6)
        assert torch.equal(y, (x.float() + m(xn).float()).to(BF))
        assert torch.equal(y[:, None], m.fused_decode_residual(x[:, None], w, 1e-6))


@pytest.mark.parametrize("nb", [5, 16, 40])
@pytest.mark.parametrize("grouped", [False, True])
def test_layer_with_norm_takes_unaligned_views(nb, grouped):
    """x or the norm weight as a view off the 16-byte grid: the result of the
    aligned copies, up to the norm's own roundings."""
    kw = dict(grouped_a=2, grouped_b=8) if grouped else {}
    m = InferenceMoCSwiGLUFFN(256, 704, 176 if grouped else 128, **kw).to("cuda", BF)
    off = lambda t: torch.cat((t.new_zeros(1), t.flatten()))[1:].view(t.shape)  # noqa: E731
    x, w = torch.randn(nb, 256, device="cuda").to(BF), torch.ones(256, device="cuda").to(BF)
    with torch.no_grad():
        assert off(x).data_ptr() % 16 and off(w).data_ptr() % 16
        for y in (m.fused_decode_residual(off(x), w, 1e-6), m.fused_decode_residual(x, off(w), 1e-6)):
            xf = x.float()
            xn = (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)).to(BF) * w
            assert torch.equal(y, x + m(xn))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, BF])
def test_after_gate_adds_a_residual_of_any_type(dtype):
    """More than 16 tokens: residual + the layer, in the sum's own type."""
    x, w = _case(20, 64, 200, 11)
    wdt = K.down_weight_t_for_decode(w[2])
    g = K.linear(x, w[0])
    res = torch.randn(20, 64, device="cuda").to(dtype)
    plain = K.global_after_gate(x, g, w[1], wdt, 50)
    got = K.global_after_gate(x, g, w[1], wdt, 50, residual=res)
    want = res + plain
    assert got.dtype == want.dtype and torch.equal(got, want)
    out = torch.empty(20, 64, dtype=BF, device="cuda")
    assert K.global_after_gate(x, g, w[1], wdt, 50, residual=res, out=out) is out
    assert torch.equal(out, want.to(BF))


@pytest.mark.parametrize("residual", [False, True])
def test_global_layer_of_more_than_2_gib_of_channels(residual):
    """More tokens than a product's operands may hold: the layer in parts."""
    nb, hidden, inter, k = 140000, 64, 8000, 8
    x, w = _case(nb, hidden, inter, 13)
    m = InferenceMoCSwiGLUFFN(hidden, inter, k).to("cuda", BF)
    for p, t in zip((m.gate_proj, m.up_proj, m.down_proj), w):
        p.weight.data.copy_(t)
    parts = slice(0, 60000), slice(60000, 120000), slice(120000, None)
    if residual:
        wdt, g = K.down_weight_t_for_decode(w[2]), K.linear(x, w[0])
        idx = torch.empty(nb, k, dtype=torch.int32, device="cuda")
        got = K.global_after_gate(x, g, w[1], wdt, k, residual=x, idx_out=idx)
        want = [K.global_after_gate(x[s], g[s], w[1], wdt, k, residual=x[s]) for s in parts]
        assert torch.equal(idx, K.topk_rows(g, k, idx_dtype=torch.int32)[1])
    else:
        assert not K.ffn_infer_fits(x, w[0], w[1], K.down_weight_t_for_decode(w[2]))
        got, want = m(x), [m(x[s]) for s in parts]
    assert torch.equal(got, torch.cat(want))
