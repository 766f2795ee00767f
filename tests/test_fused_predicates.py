"""Which modules the fused halves of a block and of a decode step stand in for:
the predicates alone, on CPU tensors that report a device (nothing is launched).
A fused half reads every operand through a bare pointer with sizes taken from
its input, so a module of another shape has to keep the stock composition."""
import pytest
import torch
import torch.nn as nn
from torch.nn.modules.module import register_module_forward_hook

from moc_amd import MoCConfig, build_model
from moc_amd.block import _own_head_dw, _own_head_dx, attention_half_ok, lm_head_ok, next_token_loss_ok
from moc_amd.ffn import block_ffn_f32_ok, block_ffn_ok
from moc_amd.inference.decode_model import DecodeConfig, DecoderModel, make_step
from moc_amd.inference.decode_model import RMSNorm as DecodeNorm
from moc_amd.model import CausalSelfAttention, RMSNorm, TransformerBlock

BF = torch.bfloat16


@pytest.fixture
def on_device(monkeypatch):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)


def _block(dtype=BF, hidden=256, inter=512):
    cfg = MoCConfig(hidden_size=hidden, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=4,
                    vocab_size=32, max_seq_len=32)
    return TransformerBlock(cfg, "moc").to(dtype)


def _linear(n_in, n_out):
    return nn.Linear(n_in, n_out, bias=False).to(BF)


def _attn_ok(blk, x):
    return attention_half_ok(x, blk.attn_norm, RMSNorm, blk.attn, CausalSelfAttention)


ATTENTION = {
    "narrow norm": lambda b: setattr(b, "attn_norm", RMSNorm(128).to(BF)),
    "broadcast norm": lambda b: setattr(b, "attn_norm", RMSNorm(1).to(BF)),
    "narrow out_proj": lambda b: setattr(b.attn, "out_proj", _linear(256, 128)),
    "out_proj of another input": lambda b: setattr(b.attn, "out_proj", _linear(128, 256)),
    "narrow qkv_proj": lambda b: setattr(b.attn, "qkv_proj", _linear(256, 512)),
    "qkv_proj of another input": lambda b: setattr(b.attn, "qkv_proj", _linear(128, 768)),
    "short sin": lambda b: setattr(b.attn, "rope_sin", b.attn.rope_sin[:8].clone()),
    "short tables": lambda b: [setattr(b.attn, n, getattr(b.attn, n)[:8].clone()) for n in ("rope_cos", "rope_sin")],
    "narrow tables": lambda b: [setattr(b.attn, n, getattr(b.attn, n)[:, :16].clone())
                                for n in ("rope_cos", "rope_sin")],
    "narrow sin": lambda b: setattr(b.attn, "rope_sin", b.attn.rope_sin[:, :16].clone()),
    "flat tables": lambda b: [setattr(b.attn, n, getattr(b.attn, n).flatten()) for n in ("rope_cos", "rope_sin")],
}


@pytest.mark.parametrize("change", list(ATTENTION))
def test_attention_half_takes_only_its_shapes(on_device, change):
    blk, x = _block(), torch.zeros(2, 16, 256, dtype=BF)
    assert _attn_ok(blk, x)
    ATTENTION[change](blk)
    assert not _attn_ok(blk, x)


def test_attention_half_takes_longer_tables(on_device):
    blk = _block()
    assert _attn_ok(blk, torch.zeros(2, 32, 256, dtype=BF)) and not _attn_ok(blk, torch.zeros(2, 33, 256, dtype=BF))


@pytest.fixture
def autocast():
    """bf16 autocast for the device type, which torch.autocast refuses to enter without one."""
    was = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
    torch.set_autocast_enabled("cuda", True)
    torch.set_autocast_dtype("cuda", BF)
    yield
    torch.set_autocast_enabled("cuda", was[0])
    torch.set_autocast_dtype("cuda", was[1])


FFN = {
    "narrow norm": lambda b, dt: setattr(b, "ffn_norm", RMSNorm(128).to(dt)),
    "broadcast norm": lambda b, dt: setattr(b, "ffn_norm", RMSNorm(1).to(dt)),
    "gate_proj of another input": lambda b, dt: setattr(b.ffn, "gate_proj", nn.Linear(128, 512, bias=False).to(dt)),
    "up_proj of another input": lambda b, dt: setattr(b.ffn, "up_proj", nn.Linear(128, 512, bias=False).to(dt)),
    "narrow up_proj": lambda b, dt: setattr(b.ffn, "up_proj", nn.Linear(256, 504, bias=False).to(dt)),
    "narrow down_proj": lambda b, dt: setattr(b.ffn, "down_proj", nn.Linear(512, 128, bias=False).to(dt)),
    "down_proj of another input": lambda b, dt: setattr(b.ffn, "down_proj", nn.Linear(504, 256, bias=False).to(dt)),
}


def _ffn_halves(blk, h):
    return block_ffn_ok(h, blk.ffn_norm.weight, blk.ffn), block_ffn_f32_ok(h, blk.ffn_norm.weight, blk.ffn)


@pytest.mark.parametrize("change", list(FFN))
def test_bf16_ffn_half_takes_only_its_shapes(on_device, change):
    blk, h = _block(), torch.zeros(2, 16, 256, dtype=BF)
    assert _ffn_halves(blk, h) == (True, False)
    FFN[change](blk, BF)
    assert _ffn_halves(blk, h) == (False, False)


@pytest.mark.parametrize("change", list(FFN))
def test_f32_ffn_half_takes_only_its_shapes(on_device, autocast, change):
    blk, h = _block(torch.float32), torch.zeros(2, 16, 256)
    assert _ffn_halves(blk, h) == (False, True)
    FFN[change](blk, torch.float32)
    assert _ffn_halves(blk, h) == (False, False)


@pytest.mark.parametrize("change", [c for c in FFN if "norm" not in c and c != "narrow down_proj"])
def test_ffn_layer_refuses_weights_that_do_not_fit(on_device, change):
    blk = _block()
    FFN[change](blk, BF)
    with pytest.raises(ValueError, match="shapes"):
        blk.ffn(torch.zeros(2, 16, 256, dtype=BF))


def test_ffn_layer_refuses_another_hidden_size(on_device):
    with pytest.raises(ValueError, match="shapes"):
        _block().ffn(torch.zeros(2, 16, 128, dtype=BF))


def _swap_instance(m, name="forward"):
    """As wrapping tools do it: the instance gets a function of its own."""
    inner = getattr(m, name)
    setattr(m, name, lambda *a, **k: inner(*a, **k))


def _swap_class(monkeypatch, cls, name="forward"):
    inner = getattr(cls, name)
    monkeypatch.setattr(cls, name, lambda *a, **k: inner(*a, **k))


@pytest.mark.parametrize("part", ["attn_norm", "attn", "attn.qkv_proj", "attn.out_proj"])
@pytest.mark.parametrize("where", ["instance", "class"])
def test_attention_half_leaves_a_replaced_forward_alone(on_device, monkeypatch, part, where):
    blk, x = _block(), torch.zeros(2, 16, 256, dtype=BF)
    m = blk.get_submodule(part)
    _swap_instance(m) if where == "instance" else _swap_class(monkeypatch, type(m))
    assert not _attn_ok(blk, x)


@pytest.mark.parametrize("part", ["norm", "lm_head"])
@pytest.mark.parametrize("where", ["instance", "class", "subclass"])
def test_lm_head_leaves_a_replaced_forward_alone(on_device, monkeypatch, part, where):
    model = nn.Module()
    model.norm, model.lm_head = RMSNorm(64).to(BF), _linear(64, 128)
    h = torch.zeros(1, 4, 64, dtype=BF)
    ok = lambda: lm_head_ok(h, model.norm, RMSNorm, model.lm_head, model.lm_head.weight)  # noqa: E731
    assert ok()
    m = getattr(model, part)
    if where == "instance":
        _swap_instance(m)
    elif where == "class":
        _swap_class(monkeypatch, type(m))
    else:
        m.__class__ = type("Own", (type(m),), {"forward": lambda self, t: t})
    assert not ok()


@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("where", ["instance", "class", "subclass"])
def test_ffn_half_leaves_a_replaced_ffn_forward_alone(on_device, monkeypatch, request, dtype, where):
    if dtype == torch.float32:
        request.getfixturevalue("autocast")
    blk, h = _block(dtype), torch.zeros(2, 16, 256, dtype=dtype)
    assert any(_ffn_halves(blk, h))
    if where == "instance":
        _swap_instance(blk.ffn)
    elif where == "class":
        _swap_class(monkeypatch, type(blk.ffn))
    else:
        blk.ffn.__class__ = type("Own", (type(blk.ffn),), {"forward": lambda self, t: t})
    assert not any(_ffn_halves(blk, h))


def test_ffn_half_takes_a_subclass_without_a_forward_of_its_own(on_device):
    blk, h = _block(), torch.zeros(2, 16, 256, dtype=BF)
    blk.ffn.__class__ = type("Named", (type(blk.ffn),), {})
    assert _ffn_halves(blk, h) == (True, False)


def _decoder():
    cfg = DecodeConfig(hidden=256, intermediate=704, heads=4, layers=1, vocab=64, k=128, max_seq=8)
    m = DecoderModel("global_moc", cfg).to(BF)
    m.allocate_cache()
    return m


@pytest.mark.parametrize("part,name", [("attn_norm", "forward"), ("attn", "forward_step"), ("attn.qkv_proj", "forward"),
                                       ("attn.out_proj", "forward")])
@pytest.mark.parametrize("where", ["instance", "class", "other"])
def test_decode_attention_leaves_a_replaced_forward_alone(on_device, monkeypatch, part, name, where):
    layer, x = _decoder().layers[0], torch.zeros(1, 1, 256, dtype=BF)
    with torch.no_grad():
        assert layer._attn_native(x)
        m = layer.get_submodule(part)
        if where == "instance":
            _swap_instance(m, name)
        elif where == "class":
            _swap_class(monkeypatch, type(m), name)
        elif isinstance(m, nn.Linear):  # a module of another kind that happens to hold a weight
            other = nn.Module()
            other.weight = m.weight
            setattr(layer.attn, part.split(".")[1], other)
        else:
            m.__class__ = type("Own", (type(m),), {})
        assert not layer._attn_native(x)


@pytest.mark.parametrize("part", ["final_norm", "lm_head"])
@pytest.mark.parametrize("where", ["instance", "class", "other"])
def test_decode_head_leaves_a_replaced_forward_alone(on_device, monkeypatch, part, where):
    model, x = _decoder(), torch.zeros(1, 1, 256, dtype=BF)
    with torch.no_grad():
        assert model._head_native(x)
        m = getattr(model, part)
        if where == "instance":
            _swap_instance(m)
        elif where == "class":
            _swap_class(monkeypatch, type(m))
        elif part == "lm_head":
            model.lm_head = nn.Sequential(m)
        else:
            m.__class__ = type("Own", (type(m),), {})
        assert not model._head_native(x)


def test_model_takes_a_head_of_another_kind():
    """A head without a weight of its own (a wrapper around the linear) is called."""
    torch.manual_seed(0)
    cfg = MoCConfig(hidden_size=64, intermediate_size=128, num_hidden_layers=0, num_attention_heads=4, vocab_size=32)
    model = build_model(cfg, "moc")
    ids = torch.randint(0, 32, (2, 8))
    want = model(ids)
    model.lm_head = nn.Sequential(model.lm_head)
    assert torch.equal(model(ids), want)


def _hook(module, kind):
    """A forward hook on the module, or one for every module; (calls, handle)."""
    seen = []
    if kind == "own":
        return seen, module.register_forward_hook(lambda m, *a: seen.append(m))
    return seen, register_module_forward_hook(lambda m, *a: seen.append(m))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("part", ["ffn_norm", "ffn"])
@pytest.mark.parametrize("kind", ["own", "every"])
def test_ffn_half_calls_hooked_modules(dtype, part, kind):
    blk = _block(dtype).cuda()
    x = torch.randn(2, 16, 256, device="cuda").to(dtype)
    m = blk.get_submodule(part)
    with torch.autocast("cuda", dtype=BF, enabled=dtype == torch.float32):
        want = blk(x)
        seen, handle = _hook(m, kind)
        try:
            got = blk(x)
        finally:
            handle.remove()
        assert sum(s is m for s in seen) == 1
        # the stock composition: bf16 roundings of the norm's and the FFN's output
        # where the fused half has none, in a stream of unit scale
        assert (got.float() - want.float()).norm() <= 2e-2 * want.float().norm()
        blk(x)
    assert sum(s is m for s in seen) == 1


@pytest.mark.gpu
def test_ffn_half_calls_a_norm_of_another_type():
    class Doubled(RMSNorm):
        def forward(self, t):
            return 2 * super().forward(t)

    blk = _block().cuda()
    x = torch.randn(2, 16, 256, device="cuda").to(BF)
    blk.ffn_norm.__class__ = Doubled
    with torch.no_grad():
        got = blk(x)
        h = x + blk.attn(blk.attn_norm(x))
        want = h + blk.ffn(2 * RMSNorm.forward(blk.ffn_norm, h))
    assert (got.float() - want.float()).norm() <= 2e-2 * want.float().norm()


@pytest.mark.parametrize("change", [
    lambda la: setattr(la, "attn_norm", DecodeNorm(1).to(BF)),
    lambda la: [setattr(la.attn, n, torch.cat([getattr(la.attn, n)] * 2)) for n in ("rope_cos", "rope_sin")],
    lambda la: setattr(la.attn, "out_proj", _linear(256, 128)),
    lambda la: setattr(la.attn, "qkv_proj", _linear(256, 512)),
    lambda la: setattr(la.attn, "v", la.attn.v[:, :, :4].clone()),
    lambda la: setattr(la.attn, "k_t", la.attn.k_t[:, :2].clone()),
], ids=["broadcast norm", "longer tables", "narrow out_proj", "narrow qkv_proj", "short v", "fewer heads"])
def test_decode_attention_takes_only_its_shapes(on_device, change):
    layer, x = _decoder().layers[0], torch.zeros(1, 1, 256, dtype=BF)
    with torch.no_grad():
        assert layer._attn_native(x)
        change(layer)
        assert not layer._attn_native(x)


@pytest.mark.parametrize("change", [
    lambda m: setattr(m, "final_norm", DecodeNorm(1).to(BF)),
    lambda m: setattr(m, "lm_head", _linear(128, 64)),
], ids=["broadcast norm", "head of another input"])
def test_decode_head_takes_only_its_shapes(on_device, change):
    model, x = _decoder(), torch.zeros(1, 1, 256, dtype=BF)
    with torch.no_grad():
        assert model._head_native(x)
        change(model)
        assert not model._head_native(x)


def test_attention_half_leaves_long_sequences_to_the_library(on_device):
    cfg = MoCConfig(hidden_size=256, intermediate_size=512, num_hidden_layers=1, num_attention_heads=4,
                    vocab_size=32, max_seq_len=8192)
    blk = TransformerBlock(cfg, "moc").to(BF)
    assert _attn_ok(blk, torch.zeros(1, 4096, 256, dtype=BF))
    assert not _attn_ok(blk, torch.zeros(1, 4097, 256, dtype=BF))


@pytest.mark.parametrize("d,vocab,own", [(512, 16384, False), (512, 24576, False), (512, 26624, True), (512, 32000, True),
                                         (576, 16384, False), (640, 20480, True), (640, 24576, False),
                                         (768, 24576, False), (768, 32000, True), (1024, 16384, True),
                                         (1536, 16384, True), (2048, 32000, True), (256, 32000, False),
                                         (1024, 8192, False)])
def test_head_weight_gradient_takes_the_engine_where_its_rounds_fill(d, vocab, own):
    """Each side is the faster one measured (_own_head_dw)."""
    assert _own_head_dw(d, vocab, 4096) == own


@pytest.mark.parametrize("p", [-1, 8, 100])
def test_decode_step_refuses_a_position_outside_the_cache(p):
    """The fused half would return NaN, where the stock composition's indexing refuses."""
    cfg = DecodeConfig(hidden=64, intermediate=176, heads=4, layers=1, vocab=64, k=32, max_seq=8)
    m = DecoderModel("dense", cfg)
    m.allocate_cache()
    step = make_step(m, "eager")
    assert step(torch.zeros(1, 1, dtype=torch.int64), 7).shape == (1, 1, 64)
    with pytest.raises(ValueError, match="position"):
        step(torch.zeros(1, 1, dtype=torch.int64), p)


@pytest.mark.gpu
@pytest.mark.parametrize("scope", ["eager", "layer_graph", "whole_graph"])
def test_decode_step_refuses_a_position_in_every_scope(scope):
    cfg = DecodeConfig(hidden=256, intermediate=704, heads=4, layers=2, vocab=64, k=128, max_seq=8)
    m = DecoderModel("global_moc", cfg).to("cuda", BF).init_weights(1)
    m.allocate_cache()
    step = make_step(m, scope)
    tok = torch.zeros(1, 1, dtype=torch.int64, device="cuda")
    assert torch.isfinite(step(tok, 7)).all()
    for p in (-1, 8):
        with pytest.raises(ValueError, match="position"):
            step(tok, p)


class _Wrapped(torch.Tensor):
    """Stands for a tensor type of its own (sharded, quantised): its storage is not what the kernels read."""


def _wrap(m, name="weight"):
    old = getattr(m, name)
    if isinstance(old, nn.Parameter):
        setattr(m, name, nn.Parameter(old.detach().as_subclass(_Wrapped)))
    else:
        setattr(m, name, old.as_subclass(_Wrapped))


@pytest.mark.parametrize("part", ["attn_norm.weight", "attn.qkv_proj.weight", "attn.out_proj.weight", "attn.rope_cos", "x"])
def test_attention_half_leaves_other_tensor_types_alone(on_device, part):
    blk, x = _block(), torch.zeros(2, 16, 256, dtype=BF)
    if part == "x":
        x = x.as_subclass(_Wrapped)
    else:
        mod, name = part.rsplit(".", 1)
        _wrap(blk.get_submodule(mod), name)
    assert not _attn_ok(blk, x)


@pytest.mark.parametrize("part", ["norm", "lm_head", "h"])
def test_lm_head_leaves_other_tensor_types_alone(on_device, part):
    norm, head, h = RMSNorm(64).to(BF), _linear(64, 128), torch.zeros(1, 4, 64, dtype=BF)
    if part == "h":
        h = h.as_subclass(_Wrapped)
    else:
        _wrap(norm if part == "norm" else head)
    assert not lm_head_ok(h, norm, RMSNorm, head, head.weight)


def test_loss_leaves_other_tensor_types_alone(on_device):
    x, labels = torch.zeros(2, 4, 64, dtype=BF), torch.zeros(2, 4, dtype=torch.int64)
    assert next_token_loss_ok(x, labels)
    assert not next_token_loss_ok(x.as_subclass(_Wrapped), labels)
    assert not next_token_loss_ok(x, labels.as_subclass(_Wrapped))


def test_decode_step_leaves_other_tensor_types_alone(on_device):
    x = torch.zeros(1, 1, 256, dtype=BF)
    with torch.no_grad():
        for part in ("attn_norm", "attn.qkv_proj", "attn.out_proj"):
            layer = _decoder().layers[0]
            _wrap(layer.get_submodule(part))
            assert not layer._attn_native(x)
        for part in ("final_norm", "lm_head"):
            model = _decoder()
            _wrap(getattr(model, part))
            assert not model._head_native(x)


def test_attention_half_leaves_operands_of_2_gib_to_the_library(on_device):
    """The engine addresses an operand with 32 bits: q/k/v rows of 1536 bytes here."""
    blk = _block()
    x = torch.zeros(1, dtype=BF).expand(43692, 32, 256)
    assert _attn_ok(blk, x[:43000]) and not _attn_ok(blk, x)


@pytest.mark.parametrize("tokens,d,vocab,dx,dw", [(32768, 256, 32000, True, False), (65536, 128, 32000, False, False),
                                                  (4096, 2048, 32000, True, True), (65536, 1024, 32000, False, False),
                                                  (2048, 4096, 262144, False, True), (2048, 4096, 131072, True, True), (2048, 4096, 524288, False, False)])
def test_head_gradients_leave_operands_of_2_gib_to_the_library(tokens, d, vocab, dx, dw):
    assert (_own_head_dx(tokens, d, vocab), _own_head_dw(d, vocab, tokens)) == (dx, dw)
