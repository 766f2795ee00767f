"""The workloads this library is timed on, each through its public entry points.

Five kinds of work, as a user's program has them:

  ffn      one MoC FFN layer's training step, forward and backward
           (build_ffn), in bf16, f32, or f32 parameters under bf16 autocast;
  block    one decoder block's training step, forward and backward
           (TransformerBlock: attention half and FFN half);
  model    one training step of a whole decoder: logits, loss, gradients
           (build_model);
  infer    inference FFN layers (InferenceMoCSwiGLUFFN): at most 16 tokens, a
           stack of layers with pre-norm and residual replayed from a HIP
           graph (each layer has its own weights, so they come from HBM); more
           tokens, one layer called as it is;
  decode   a whole decoder (DecoderModel): one token with a filled KV cache
           through the captured step, or the prompt.

Weights are N(0, 0.02) and activations N(0, 1), the scales of an initialised
model behind its norms.  Where layers are stacked, or a block adds to a residual
stream, the stream starts at unit scale and the projections that write to it
are N(0, 0.01 / sqrt(2 layers)), so that a layer adds a small part of what the
stream holds, as in a trained decoder: a stream of random layers at full scale
amplifies each rounding layer by layer, which a trained one does not.  Sizes are those of the presets and of the benchmark,
and what lies between and around them: odd intermediate sizes, ragged token
counts, one token.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from moc_amd import MoCConfig, build_ffn, build_model
from moc_amd.inference.decode_model import DecodeConfig, DecoderModel, make_step
from moc_amd.inference.inference_ffn import InferenceMoCSwiGLUFFN
from moc_amd.model import TransformerBlock

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
EPS = 1e-6
VOCAB = 32000


def listed():
    return [
        # A 60m layer in full precision, as in a debugging or parity run: short
        # launches, the host and the launch count matter as much as the kernels.
        dict(name="ffn_f32_60m", kind="ffn", dtype="f32", ffn_type="moc", tokens=512, hidden=512, inter=1376,
             k=256),
        # A 130m layer with gate checkpointing on 8 x 1024 tokens.
        dict(name="ffn_gcp_130m", kind="ffn", dtype="bf16", ffn_type="moc_gcp", tokens=8192, hidden=768,
             inter=2048, k=384),
        # The benchmark's layer: 1b, 64 x 256 tokens, an intermediate size
        # whose rows are not 16-byte aligned.
        dict(name="ffn_moc_1b", kind="ffn", dtype="bf16", ffn_type="moc", tokens=16384, hidden=2048, inter=5461,
             k=1024),
        # A 350m layer, structured 2:8 selection, on a short ragged batch (the
        # last batch of an epoch, a small fine-tuning batch).
        dict(name="ffn_28_350m_ragged", kind="ffn", dtype="bf16", ffn_type="moc_2_8", tokens=1000, hidden=1024,
             inter=2736, k=512),
        # A 350m decoder block in a bf16 training step of 16 x 256 tokens.
        dict(name="block_gcp_350m", kind="block", dtype="bf16", ffn_type="moc_gcp", batch=16, seq=256,
             hidden=1024, heads=16, inter=2736, k=512),
        # A whole 60m model's step with f32 parameters under bf16 autocast, the
        # setting the presets are trained in.
        dict(name="model_60m_autocast", kind="model", dtype="autocast", ffn_type="moc", batch=16, seq=256,
             hidden=512, heads=8, layers=8, inter=1376, k=256),
        # Decode, one token: eight 1b FFN layers, global Top-K selection.
        dict(name="infer_global_b1", kind="infer", grouped=False, tokens=1, hidden=2048, inter=5461, k=1024,
             layers=8),
        # Decode, a batch of 16: eight 1b FFN layers, 2:8 selection.
        dict(name="infer_28_b16", kind="infer", grouped=True, tokens=16, hidden=2048, inter=5464, k=1366,
             layers=8),
        # A large decode batch, or a short prompt: more tokens than the decode
        # kernels take, far fewer than a prefill's.
        dict(name="infer_global_200", kind="infer", grouped=False, tokens=200, hidden=2048, inter=5461, k=1024,
             layers=1),
        # The same for 2:8 at a ragged serving batch.
        dict(name="infer_28_48", kind="infer", grouped=True, tokens=48, hidden=2048, inter=5464, k=1366,
             layers=1),
        # 2:8 prefill of 4096 tokens.
        dict(name="infer_28_4096", kind="infer", grouped=True, tokens=4096, hidden=2048, inter=5464, k=1366,
             layers=1),
        # A 24-layer decoder's next token after a prompt of 128: the benchmark's
        # end-to-end decode.
        dict(name="decode_global_24", kind="decode", phase="step", row="global_moc", hidden=2048, heads=16,
             inter=5464, k=1024, layers=24, prompt=128, max_seq=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["ffn", "block", "model", "infer", "decode"], [35, 12, 5, 36, 12])[0]
    types = ["moc", "moc_gcp", "moc_2_8", "moc_post_silu_abs"]
    if kind == "ffn":
        dtype = rng.choices(["bf16", "autocast", "f32"], [6, 2, 2])[0]
        hidden = 64 * _log(rng, 4, 16 if dtype == "f32" else 32)
        inter = int(hidden * rng.uniform(2.0, 2.66))
        return dict(kind=kind, dtype=dtype, ffn_type=rng.choice(types),
                    tokens=_log(rng, 16, 1024 if dtype == "f32" else 16384), hidden=hidden, inter=inter,
                    k=int(hidden * rng.uniform(0.3, 0.7)))
    if kind in ("block", "model"):
        heads = _log(rng, 4, 16) if kind == "block" else 8
        hidden = 64 * heads
        seq = _log(rng, 32, 256)
        return dict(kind=kind, dtype=rng.choice(["bf16", "autocast"]), ffn_type=rng.choice(types),
                    batch=max(1, _log(rng, 64, 4096) // seq), seq=seq, hidden=hidden, heads=heads,
                    inter=8 * int(hidden * rng.uniform(2.0, 2.75) / 8), k=hidden // 2,
                    **(dict(layers=rng.randint(2, 8)) if kind == "model" else {}))
    if kind == "infer":
        grouped = rng.random() < 0.5
        tokens = _log(rng, 1, 4096)
        hidden = 128 * _log(rng, 4, 32 if tokens <= 512 else 16)
        inter = int(hidden * rng.uniform(2.0, 2.67))
        if grouped:
            inter = inter // 8 * 8
        return dict(kind=kind, grouped=grouped, tokens=tokens, hidden=hidden, inter=inter,
                    k=inter // 4 if grouped else int(hidden * rng.uniform(0.3, 0.7)),
                    layers=rng.randint(4, 8) if tokens <= 16 else 1)
    hidden = 256 * rng.choice([2, 4, 8])
    prompt = rng.randint(8, 300)
    row = rng.choice(["global_moc", "moc_2_8"])
    return dict(kind=kind, phase=rng.choice(["step", "step", "prompt"]), row=row, hidden=hidden,
                heads=hidden // rng.choice([64, 128]), inter=8 * int(hidden * rng.uniform(2.0, 2.67) / 8),
                k=hidden // 2, layers=rng.randint(2, 24), prompt=prompt, max_seq=prompt + rng.randint(1, 128))


# ------------------------------------------------------------------- prepare
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, shape, std=1.0, dtype=F32):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _fill(module, gen, depth=None):
    """N(0, 0.02) projections, norm weights around one; in a stack of `depth`
    layers the projections that write to the residual stream are smaller."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if p.dim() == 1:
                p.copy_(1 + _normal(gen, p.shape, 0.05))
            elif "emb" in name:
                p.copy_(_normal(gen, p.shape))
            else:
                to_stream = depth and ("out_proj" in name or "down_proj" in name)
                p.copy_(_normal(gen, p.shape, 0.01 / math.sqrt(2 * depth) if to_stream else 0.02))
    return module


def _config(case):
    return MoCConfig(hidden_size=case["hidden"], intermediate_size=case["inter"],
                     num_hidden_layers=case.get("layers", 1), num_attention_heads=case["heads"], vocab_size=VOCAB,
                     k=case["k"])


def _infer_layers(case, gen):
    grouped = dict(grouped_a=2, grouped_b=8) if case["grouped"] else {}
    with torch.device("cuda"):
        ffns = [InferenceMoCSwiGLUFFN(case["hidden"], case["inter"], case["k"], **grouped).to(BF16)
                for _ in range(case["layers"])]
    for f in ffns:
        _fill(f, gen, 24 if case["tokens"] <= 16 else None)  # some of 24 layers
    norms = [1 + _normal(gen, (case["hidden"],), 0.05) for _ in ffns]
    return ffns, [n.to(BF16) for n in norms]


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    dtype = BF16 if case.get("dtype", "bf16") == "bf16" else F32
    st = {"case": case}
    if kind == "ffn":
        with torch.device("cuda"):
            ffn = build_ffn(case["hidden"], case["inter"], case["ffn_type"], k=case["k"])
        st["module"] = _fill(ffn, gen).to(dtype)
        shape = (case["tokens"], case["hidden"])
    elif kind == "block":
        with torch.device("cuda"):
            block = TransformerBlock(_config(case), case["ffn_type"])
        st["module"] = _fill(block, gen, 24).to(dtype)  # one of 24 layers
        shape = (case["batch"], case["seq"], case["hidden"])
    if kind in ("ffn", "block"):
        st["x"] = _normal(gen, shape, 1.0, dtype).requires_grad_()
        # the gradient that arrives at a layer's output, in its output's type
        out_type = F32 if case["dtype"] == "f32" or (kind == "block" and dtype == F32) else BF16
        st["dy"] = _normal(gen, shape, 1.0, out_type)
    elif kind == "model":
        with torch.device("cuda"):
            model = build_model(_config(case), case["ffn_type"])
        st["module"] = _fill(model, gen, 24).to(dtype)
        st["ids"] = torch.randint(0, VOCAB, (case["batch"], case["seq"]), generator=gen, device="cuda")
    elif kind == "infer":
        ffns, norms = _infer_layers(case, gen)
        x = _normal(gen, (case["tokens"], case["hidden"]), 1.0, BF16)
        st.update(ffns=ffns, norms=norms, x=x)
        if case["tokens"] <= 16:
            st["graph"], st["in"], st["out"] = _stack_graph(ffns, norms, x)
    else:
        cfg = DecodeConfig(hidden=case["hidden"], intermediate=case["inter"], heads=case["heads"],
                           layers=case["layers"], vocab=VOCAB, k=case["k"], max_seq=case["max_seq"])
        with torch.device("cuda"):
            model = DecoderModel(case["row"], cfg).to(BF16)
        _fill(model, gen, 24)
        model.allocate_cache()
        ids = torch.randint(0, VOCAB, (1, case["prompt"] + 1), generator=gen, device="cuda")
        st.update(model=model, prompt=ids[:, :-1].contiguous(), token=ids[:, -1:].contiguous())
        if case["phase"] == "step":
            st["step"] = make_step(model, "whole_graph")
            model.reset_cache()
            model.forward_prompt(st["prompt"])
    return st


def _stack_graph(ffns, norms, x):
    """h <- h + FFN(RMSNorm(h)) over the layers, captured in a HIP graph."""
    buf = x.clone()

    @torch.no_grad()
    def stack():
        h, outs = buf, []
        for ffn, norm in zip(ffns, norms):
            h = ffn.fused_decode_residual(h, norm, EPS)
            outs.append(h)
        return outs

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            stack()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = stack()
    return graph, buf, outs


# ----------------------------------------------------------------------- run
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("ffn", "block"):
        mod, x = st["module"], st["x"]
        mod.zero_grad(set_to_none=True)
        x.grad = None
        with torch.autocast("cuda", dtype=BF16, enabled=case["dtype"] == "autocast"):
            y = mod(x)
        y.backward(st["dy"])
        return [y, x.grad, [p.grad for p in mod.parameters()]]
    if kind == "model":
        mod = st["module"]
        mod.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=BF16, enabled=case["dtype"] == "autocast"):
            logits, loss = mod(st["ids"], labels=st["ids"])
        loss.backward()
        return [logits, loss, [p.grad for p in mod.parameters()]]
    if kind == "infer":
        if "graph" in st:
            st["in"].copy_(st["x"])
            st["graph"].replay()
            return st["out"]
        with torch.no_grad():
            return [st["ffns"][0](st["x"])]
    model = st["model"]
    if case["phase"] == "prompt":
        logits = model.forward_prompt(st["prompt"])
    else:
        logits = st["step"](st["token"], case["prompt"])
    return [logits, [[la.attn.k_t, la.attn.v] for la in model.layers]]


# ---------------------------------------------------------------------- work
def _ffn_train_work(t, d, i, k, act, par):
    """G for every channel; U, D and the six backward products only where a
    channel is selected.  x, dy, y, dx; weights read, gradients written."""
    return (4 * t * d * act + 6 * d * i * par, 2.0 * t * d * i + 16.0 * t * d * k)


def work(case):
    kind = case["kind"]
    d, i = case["hidden"], case["inter"]
    grouped = case.get("grouped") or case.get("ffn_type") == "moc_2_8" or case.get("row") == "moc_2_8"
    k = 2 * (i // 8) + min(2, i % 8) if grouped else case["k"]
    if kind == "infer" or kind == "decode":
        t = case["tokens"] if kind == "infer" else case["prompt"] if case["phase"] == "prompt" else 1
        union = i * (1.0 - (1.0 - k / i) ** t)  # channels that some token selects
        nbytes = 2 * d * (i + 2 * union) + 2 * 2 * t * d
        flops = 2.0 * t * d * i + 4.0 * t * d * k
        if kind == "decode":
            keys = case["prompt"] + (case["phase"] == "step")
            nbytes += 2 * 4 * d * d + 2 * 2 * d * keys
            flops += 8.0 * t * d * d + 4.0 * t * d * (keys if t == 1 else keys / 2)
        nbytes, flops = nbytes * case["layers"], flops * case["layers"]
        if kind == "decode":
            nbytes += 2 * d * VOCAB + 2 * t * VOCAB
            flops += 2.0 * t * d * VOCAB
        return {"bytes": nbytes, "flops": flops}
    par = 2 if case["dtype"] == "bf16" else 4
    t = case["tokens"] if kind == "ffn" else case["batch"] * case["seq"]
    # autocast: x and dx of a layer in f32, y and dy in bf16
    act = {"bf16": 2, "f32": 4, "autocast": 3}[case["dtype"]]
    nbytes, flops = _ffn_train_work(t, d, i, k, act, par)
    if kind in ("block", "model"):
        nbytes += 2 * 4 * d * d * par
        flops += 3 * (8.0 * t * d * d + 2.0 * t * d * case["seq"])
    if kind == "model":
        nbytes = nbytes * case["layers"] + 3 * VOCAB * d * par + 2 * t * VOCAB * 2
        flops = flops * case["layers"] + 6.0 * t * d * VOCAB
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # A channel whose gate score lies within a rounding of the row's k-th can
    # be selected by one correct implementation and not by another.  One such
    # channel is 2e-3 of a 512-token layer's norm, and a single row or gradient
    # entry can change as a whole ("max").
    kind = case["kind"]
    if case.get("dtype") == "f32":
        return {"rel": 2e-3, "max": 0.99}
    if kind == "ffn" or (kind == "infer" and case["tokens"] > 16):
        return {"rel": 1e-2, "max": 0.99}  # bf16 results: 4e-3 off 64 bits
    # a rounding of the residual stream moves the next layers' selections
    return {"rel": 3e-2, "max": 0.99}


# --------------------------------------------------------------------- exact
def _select(scores, k, grouped):
    """Boolean mask of the selected channels: value descending, then channel."""
    t, i = scores.shape
    if grouped:
        pad = F.pad(scores.float(), (0, -i % 8), value=-math.inf).reshape(t, -1, 8)
        order = torch.sort(pad, dim=-1, descending=True, stable=True).indices[..., :2]
        return torch.zeros_like(pad, dtype=torch.bool).scatter_(-1, order, True).reshape(t, -1)[:, :i]
    order = torch.sort(scores.float(), dim=-1, descending=True, stable=True).indices[:, :k]
    return torch.zeros_like(scores, dtype=torch.bool).scatter_(-1, order, True)


def _ffn64(x, wg, wu, wd, k, kind, dt):
    """The layer in 64 bits; channels are selected by the gate scores as the
    path holds them (rounded to dt)."""
    g = x @ wg.t()
    score = g.detach().to(dt)
    if kind == "moc_post_silu_abs":
        score = F.silu(score.float()).to(dt).abs()
    mask = _select(score, k, kind == "moc_2_8")
    return (F.silu(g) * (x @ wu.t()) * mask) @ wd.t()


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _rope64(x, pos, theta=10000.0):
    hd = x.shape[-1]
    inv = theta ** (-torch.arange(0, hd, 2, dtype=F64, device=x.device) / hd)
    ang = pos.to(F64)[:, None] * inv
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), dim=-1).flatten(-2)


def _heads64(x, w_qkv, heads):
    b, n, d = x.shape
    q, k, v = (x @ w_qkv.t()).view(b, n, 3, heads, d // heads).permute(2, 0, 3, 1, 4)
    pos = torch.arange(n, device=x.device)
    return _rope64(q, pos), _rope64(k, pos), v


def _attend64(q, k, v, w_out):
    b, h, n, hd = q.shape
    s = q @ k.transpose(-1, -2) / math.sqrt(hd)
    s = s + torch.full((n, n), -math.inf, dtype=F64, device=q.device).triu(1)
    y = torch.softmax(s, -1) @ v
    return y.permute(0, 2, 1, 3).reshape(b, n, h * hd) @ w_out.t()


def _block64(x, p, prefix, case):
    """p: named parameters in 64 bits."""
    n1, n2, wq, wo, wg, wu, wd = (p[prefix + n + ".weight"] for n in (
        "attn_norm", "ffn_norm", "attn.qkv_proj", "attn.out_proj", "ffn.gate_proj", "ffn.up_proj", "ffn.down_proj"))
    h = x + _attend64(*_heads64(_norm64(x, n1), wq, case["heads"]), wo)
    xn = _norm64(h, n2).flatten(0, 1)
    return h + _ffn64(xn, wg, wu, wd, case["k"], case["ffn_type"], BF16).view(h.shape)


class _Operand(torch.autograd.Function):
    """A product's operand as autocast casts it; gradients pass unchanged."""

    @staticmethod
    def forward(ctx, x):
        return x.to(BF16).to(F64)

    @staticmethod
    def backward(ctx, g):
        return g


def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind in ("infer", "decode"):
        with torch.no_grad():
            return _exact_infer(case, st) if kind == "infer" else _exact_decode(case, st)
    named = {n: p.detach().to(F64).requires_grad_() for n, p in st["module"].named_parameters()}
    cast = _Operand.apply if case["dtype"] == "autocast" else lambda t: t
    used = {n: cast(p) if p.dim() > 1 and "tok_emb" not in n else p for n, p in named.items()}
    if kind == "model":
        h = used["tok_emb.weight"][st["ids"]]
        for n in range(case["layers"]):
            h = _block64(h, used, "blocks.%d." % n, case)
        logits = _norm64(h, used["norm.weight"]) @ used["lm_head.weight"].t()
        loss = F.cross_entropy(logits[:, :-1].flatten(0, 1), st["ids"][:, 1:].flatten())
        loss.backward()
        return [logits, loss, [p.grad for p in named.values()]]
    x = st["x"].detach().to(F64).requires_grad_()
    if kind == "ffn":
        dt = F32 if case["dtype"] == "f32" else BF16
        y = _ffn64(cast(x), used["gate_proj.weight"], used["up_proj.weight"], used["down_proj.weight"], case["k"],
                   case["ffn_type"], dt)
    else:
        y = _block64(x, used, "", case)
    y.backward(st["dy"].to(F64))
    return [y, x.grad, [p.grad for p in named.values()]]


def _infer64(ffn, x, k, grouped):
    w = [p.weight.to(F64) for p in (ffn.gate_proj, ffn.up_proj, ffn.down_proj)]
    return _ffn64(x, *w, k, "moc_2_8" if grouped else "moc", BF16)


def _exact_infer(case, st):
    h = st["x"].to(F64)
    if case["tokens"] > 16:
        return [_infer64(st["ffns"][0], h, case["k"], case["grouped"])]
    outs = []
    for ffn, norm in zip(st["ffns"], st["norms"]):
        h = h + _infer64(ffn, _norm64(h, norm.to(F64)), case["k"], case["grouped"])
        outs.append(h)
    return outs


def _exact_decode(case, st):
    model = st["model"]
    ids = torch.cat((st["prompt"], st["token"]), 1) if case["phase"] == "step" else st["prompt"]
    h = model.embed.weight.to(F64)[ids]
    b, n, d = h.shape
    caches = []
    for la in model.layers:
        q, k, v = _heads64(_norm64(h, la.attn_norm.weight.to(F64)), la.attn.qkv_proj.weight.to(F64), case["heads"])
        k_t, cv = (torch.zeros(t.shape, dtype=F64, device=h.device) for t in (la.attn.k_t, la.attn.v))
        k_t[..., :n], cv[:, :, :n] = k.transpose(-1, -2), v
        caches.append([k_t, cv])
        h = h + _attend64(q, k, v, la.attn.out_proj.weight.to(F64))
        xn = _norm64(h, la.ffn_norm.weight.to(F64)).flatten(0, 1)
        h = h + _infer64(la.ffn, xn, case["inter"] // 4 if case["row"] == "moc_2_8" else case["k"],
                         case["row"] == "moc_2_8").view(h.shape)
    if case["phase"] == "step":
        h = h[:, -1:]
    return [_norm64(h, model.final_norm.weight.to(F64)) @ model.lm_head.weight.to(F64).t(), caches]
