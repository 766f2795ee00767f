"""The fused one-token attention half (K.decode_attention) against the stock
composition's rounding points in 64 bits, and the decoder step that uses it."""
import math

import pytest
import torch

from moc_amd import kernels as K
from moc_amd.inference.decode_model import DecodeConfig, DecoderModel, make_step, rope_tables

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _inputs(hidden, heads, max_seq, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).to(BF)  # noqa: E731
    dim = hidden // heads
    cos, sin = (t.to("cuda", BF) for t in rope_tables(dim, max_seq))
    return dict(x=r(1, hidden), norm=1 + r(hidden, std=0.1), wqkv=r(3 * hidden, hidden, std=hidden ** -0.5),
                wout=r(hidden, hidden, std=hidden ** -0.5), cos=cos, sin=sin, k_t=r(heads, dim, max_seq),
                v=r(heads, max_seq, dim))


def _reference(t, pos, scale):
    """(y, k, v, largest |v| seen) with bf16 where the stock composition
    stores bf16 results of sums."""
    bf = lambda a: a.to(BF).double()  # noqa: E731
    heads, dim, _ = t["k_t"].shape
    x = t["x"].float()
    xn = (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)).to(BF) * t["norm"]
    q, k, v = bf(xn.double() @ t["wqkv"].double().t()).view(3, heads, dim)
    c, s = t["cos"][pos].double(), t["sin"][pos].double()
    rot = lambda a: bf(torch.stack((a[..., 0::2] * c - a[..., 1::2] * s,  # noqa: E731
                                    a[..., 0::2] * s + a[..., 1::2] * c), -1).flatten(-2))
    q, k = rot(q), rot(k)
    kk = torch.cat((t["k_t"][:, :, :pos].double(), k[:, :, None]), 2)
    vv = torch.cat((t["v"][:, :pos].double(), v[:, None]), 1)
    p = torch.softmax((q[:, None] @ kk) * scale, -1)
    o = bf((p @ vv).reshape(1, -1))
    y = bf(bf(o @ t["wout"].double().t()) + t["x"].double())
    return y, k, v, vv.abs().amax(dim=1).reshape(1, -1)


@pytest.mark.parametrize("hidden,heads,max_seq", [(64, 8, 3), (96, 4, 17), (512, 8, 255), (768, 3, 256),
                                                  (1024, 16, 700), (2048, 16, 257), (4096, 32, 2048)])
@pytest.mark.parametrize("where", ["first", "middle", "last"])
def test_against_composition(hidden, heads, max_seq, where):
    t = _inputs(hidden, heads, max_seq, hidden + max_seq)
    pos = {"first": 0, "middle": max_seq // 2, "last": max_seq - 1}[where]
    scale = 1.0 / math.sqrt(hidden // heads)
    y_ref, k_ref, v_ref, vmax = _reference(t, pos, scale)
    k0, v0 = t["k_t"].clone(), t["v"].clone()
    args = [t[n] for n in ("x", "norm")] + [1e-6] + [t[n] for n in ("wqkv", "wout", "cos", "sin")]
    y = K.decode_attention(*args, torch.tensor(pos, device="cuda"), t["k_t"], t["v"], scale)
    # the cache: the new position within an ulp (the projection, then RoPE,
    # each one rounding), the rest untouched
    for new, ref in ((t["k_t"][:, :, pos], k_ref), (t["v"][:, pos], v_ref)):
        assert ((new.double() - ref).abs() <= 2.0 ** -6 * ref.abs() + 2.0 ** -8).all()
    t["k_t"][:, :, pos], t["v"][:, pos] = k0[:, :, pos], v0[:, pos]
    assert torch.equal(t["k_t"], k0) and torch.equal(t["v"], v0)
    # y: its own rounding, and the attention output's (2^-6 of the largest V
    # covers an ulp of o and of the scores' q and k) through out_proj
    bound = 2.0 ** -7 * y_ref.abs() + 2.0 ** -6 * vmax @ t["wout"].double().abs().t() / 4 + 2.0 ** -8
    assert ((y.double() - y_ref).abs() <= bound).all()
    assert (y.double() - y_ref).norm() <= 6e-3 * y_ref.norm()


@pytest.mark.parametrize("pos", [-1, 40])
def test_position_outside_the_cache(pos):
    t = _inputs(256, 4, 40, 3)
    k0, v0 = t["k_t"].clone(), t["v"].clone()
    args = [t[n] for n in ("x", "norm")] + [1e-6] + [t[n] for n in ("wqkv", "wout", "cos", "sin")]
    y = K.decode_attention(*args, torch.tensor(pos, device="cuda"), t["k_t"], t["v"], 0.125)
    assert torch.isnan(y).all() and torch.equal(t["k_t"], k0) and torch.equal(t["v"], v0)


@pytest.mark.parametrize("row", ["global_moc", "moc_2_8", "dense"])
@pytest.mark.parametrize("hidden,heads", [(256, 4), (512, 4)])
def test_step_matches_the_unfused_model(row, hidden, heads):
    """Logits and caches of single-token steps, eager and replayed, against
    the stock composition on the same weights."""
    cfg = DecodeConfig(hidden=hidden, intermediate=704, heads=heads, layers=2, vocab=500, k=hidden // 2, max_seq=30)
    ms = [DecoderModel(row, cfg).to("cuda", BF).init_weights(5) for _ in range(2)]
    ms[1].fuse_head = False
    for la in ms[1].layers:
        la.fuse_attn = False
    prompt = torch.randint(0, 500, (1, 20), generator=torch.Generator().manual_seed(6)).cuda()
    for m in ms:
        m.allocate_cache()
        # The stream at unit scale: a branch (RMS about 0.1 here) adds its bf16
        # roundings, and the channels they move across the selection's
        # threshold (about one in 50 of the branch), to a stream ten times its
        # size: 2 layers of 2e-3 each and the stream's own 2^-9 a sum, below
        # 1e-2 in all, doubled for the LM head's input.  At init_weights' 0.02
        # the branches are the stream and the same roundings are 2.3e-2 of it.
        m.embed.weight.data.mul_(50)
    with torch.no_grad():
        one = torch.zeros(1, 1, hidden, dtype=BF, device="cuda")
        assert [m.layers[0]._attn_native(one) for m in ms] == [True, False]
    ref_step, eager, graph = make_step(ms[1], "eager"), make_step(ms[0], "eager"), make_step(ms[0], "whole_graph")
    outs = []
    for m, step in ((ms[1], ref_step), (ms[0], eager), (ms[0], graph)):
        m.reset_cache()
        m.forward_prompt(prompt)
        outs.append([step(prompt[:, i:i + 1], 20 + i).clone() for i in range(4)])
        outs[-1] += [la.attn.k_t.clone() for la in m.layers] + [la.attn.v.clone() for la in m.layers]
    for ref, a, b in zip(*outs):
        assert torch.equal(a, b)
        assert (a.float() - ref.float()).norm() <= 2e-2 * ref.float().norm()


def test_hooks_keep_the_stock_path():
    cfg = DecodeConfig(hidden=256, intermediate=704, heads=4, layers=1, vocab=100, k=128, max_seq=8)
    m = DecoderModel("global_moc", cfg).to("cuda", BF).init_weights(5)
    m.allocate_cache()
    seen = []
    m.layers[0].attn.out_proj.register_forward_hook(lambda *a: seen.append(1))
    make_step(m, "eager")(torch.zeros(1, 1, dtype=torch.int64, device="cuda"), 0)
    assert seen


def test_unaligned_token_keeps_the_stock_path():
    cfg = DecodeConfig(hidden=256, intermediate=704, heads=4, layers=1, vocab=100, k=128, max_seq=8)
    m = DecoderModel("global_moc", cfg).to("cuda", BF).init_weights(6)
    m.allocate_cache()
    layer, pos = m.layers[0], torch.tensor(0, device="cuda")
    x = torch.randn(1, 1, 256, device="cuda").to(BF)
    off = torch.cat((x.new_zeros(1), x.flatten()))[1:].view(x.shape)
    with torch.no_grad():
        assert layer._attn_native(x) and not layer._attn_native(off)
        got = layer.forward_step(off, pos)
        layer.fuse_attn = False
        assert torch.equal(got, layer.forward_step(x, pos))
