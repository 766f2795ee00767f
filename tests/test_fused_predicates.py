"""Which modules the fused halves of a block and of a decode step stand in for:
the predicates alone, on CPU tensors that report a device (nothing is launched).
A fused half reads every operand through a bare pointer with sizes taken from
its input, so a module of another shape has to keep the stock composition."""
import pytest
import torch
import torch.nn as nn

from moc_amd import MoCConfig
from moc_amd.block import attention_half_ok
from moc_amd.ffn import block_ffn_f32_ok, block_ffn_ok
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
