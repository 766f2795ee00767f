"""The model's last steps, final norm with LM head and next-token loss, against
64 bits and the stock composition."""
import pytest
import torch
import torch.nn.functional as F

from moc_amd import MoCConfig, build_model
from moc_amd.block import lm_head, lm_head_ok, next_token_loss, next_token_loss_ok
from moc_amd.model import RMSNorm

pytestmark = pytest.mark.gpu
BF, F64 = torch.bfloat16, torch.float64


@pytest.mark.parametrize("batch,seq,vocab", [(1, 2, 8), (3, 5, 4096), (2, 33, 4104), (2, 9, 32000), (1, 3, 65536),
                                             (4, 64, 1000)])
@pytest.mark.parametrize("autocast", [True, False])
def test_loss_and_gradient(batch, seq, vocab, autocast):
    g = torch.Generator(device="cuda").manual_seed(batch * seq + vocab)
    x = (3 * torch.randn(batch, seq, vocab, generator=g, device="cuda")).to(BF)
    labels = torch.randint(0, vocab, (batch, seq), generator=g, device="cuda")
    if seq > 2:
        labels[0, 1] = -100
    if batch > 2:
        labels[1] = -100
    x.requires_grad_()
    assert next_token_loss_ok(x, labels)
    with torch.autocast("cuda", dtype=BF, enabled=autocast):
        loss = next_token_loss(x, labels)
        stock = F.cross_entropy(x[:, :-1].flatten(0, 1), labels[:, 1:].flatten(), ignore_index=-100)
    assert loss.dtype == stock.dtype
    xd = x.detach().to(F64).requires_grad_()
    ref = F.cross_entropy(xd[:, :-1].flatten(0, 1), labels[:, 1:].flatten(), ignore_index=-100)
    # f32: expf, logf and a sum of vocab terms a row, then a 64-bit mean
    tol = 2e-6 if loss.dtype == torch.float32 else 2.0 ** -8
    assert abs(loss.item() - ref.item()) <= tol * max(1.0, abs(ref.item()))
    grad = torch.autograd.grad(loss, x, torch.tensor(0.7, dtype=loss.dtype, device="cuda"))[0]
    want = torch.autograd.grad(ref, xd, torch.tensor(0.7, dtype=loss.dtype).to("cuda", F64))[0]
    # its bf16 rounding; exp(x - lse) - 1 at the label cancels f32 values near 1
    assert ((grad.to(F64) - want).abs() <= 2.0 ** -8 * want.abs() + 2e-6 / (batch * (seq - 1))).all()
    assert (grad[:, -1] == 0).all()


@pytest.mark.parametrize("autocast", [True, False])
@pytest.mark.parametrize("batch,seq,vocab", [(1, 2, 8), (3, 5, 4104), (2, 9, 32000), (1, 3, 65536)])
def test_logits_may_change_between_loss_and_backward(batch, seq, vocab, autocast):
    """The gradient is that of the logits the loss saw, as with the stock loss,
    which keeps its own log-probabilities."""
    g = torch.Generator(device="cuda").manual_seed(vocab)
    leaf = torch.randn(batch, seq, vocab, generator=g, device="cuda").to(BF).requires_grad_()
    labels = torch.randint(0, vocab, (batch, seq), generator=g, device="cuda")
    labels[0, 1] = -100
    if seq * batch == 2:
        labels[0, 1] = 3
    x, y = leaf * 3, leaf * 3
    with torch.autocast("cuda", dtype=BF, enabled=autocast):
        a, b = next_token_loss(x, labels), next_token_loss(y, labels)
    with torch.no_grad():
        x.div_(0.7)
        x[..., 0] = -float("inf")
    want, = torch.autograd.grad(b, leaf)
    for _ in range(2):
        got, = torch.autograd.grad(a, leaf, retain_graph=True)
        assert torch.equal(got, want)


def test_loss_without_gradient_keeps_no_copy():
    x = torch.randn(4, 64, 32000, device="cuda").to(BF)
    labels = torch.randint(0, 32000, (4, 64), device="cuda")
    with torch.no_grad():
        next_token_loss(x, labels)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        next_token_loss(x, labels)
    assert torch.cuda.max_memory_allocated() - base < x.numel()


def test_all_ignored_and_bad_labels_are_nan():
    x = torch.randn(2, 4, 64, device="cuda").to(BF)
    assert torch.isnan(next_token_loss(x, torch.full((2, 4), -100, device="cuda")))
    labels = torch.zeros(2, 4, dtype=torch.int64, device="cuda")
    labels[1, 2] = 64
    assert torch.isnan(next_token_loss(x, labels))


def test_bad_label_gradient_is_nan():
    """A label outside the vocabulary: the gradient of its position is NaN, not
    that of a row without a label; the other rows keep theirs."""
    x = torch.randn(2, 4, 64, device="cuda").to(BF).requires_grad_()
    labels = torch.zeros(2, 4, dtype=torch.int64, device="cuda")
    labels[1, 2], labels[0, 1] = 64, -1
    grad, = torch.autograd.grad(next_token_loss(x, labels), x)
    bad = torch.zeros(2, 4, dtype=torch.bool, device="cuda")
    bad[1, 1] = bad[0, 0] = True
    assert torch.isnan(grad[bad]).all() and torch.isfinite(grad[~bad]).all()


def test_infinite_logits():
    x = torch.zeros(1, 3, 16, device="cuda").to(BF)
    x[0, 0, 3] = -float("inf")
    labels = torch.tensor([[0, 1, 2]], device="cuda")
    ref = F.cross_entropy(x.float()[:, :-1].flatten(0, 1), labels[:, 1:].flatten())
    assert abs(next_token_loss(x, labels).item() - ref.item()) < 2e-2
    x[0, 0, 3] = float("inf")  # inf - inf, as in the stock loss
    assert torch.isnan(next_token_loss(x, labels))


def test_second_derivative():
    x = torch.randn(2, 4, 64, device="cuda").to(BF).requires_grad_()
    labels = torch.randint(0, 64, (2, 4), device="cuda")
    v = torch.randn(2, 4, 64, device="cuda").to(BF)

    def hv(loss):
        return torch.autograd.grad((torch.autograd.grad(loss, x, create_graph=True)[0] * v).sum(), x)[0]

    with torch.autocast("cuda", dtype=BF):
        got = hv(next_token_loss(x, labels))
    xd = x.detach().to(F64).requires_grad_()
    loss = F.cross_entropy(xd[:, :-1].flatten(0, 1), labels[:, 1:].flatten())
    gd = torch.autograd.grad(loss, xd, create_graph=True)[0]
    want = torch.autograd.grad((gd * v.to(F64)).sum(), xd)[0]
    # bf16 roundings of the first gradient's product with v, of its cotangent
    # and of the result, each 2^-9 of its value; the cotangent's difference from
    # its mean cancels part of it
    assert (got.to(F64) - want).norm() <= 4 * 2.0 ** -9 * want.norm()


@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_model_uses_it(dtype):
    torch.manual_seed(1)
    cfg = MoCConfig(hidden_size=128, intermediate_size=344, num_hidden_layers=2, num_attention_heads=2,
                    vocab_size=1000, max_seq_len=64)
    m = build_model(cfg, "moc").to("cuda", dtype)
    ids = torch.randint(0, 1000, (3, 40), device="cuda")
    with torch.autocast("cuda", dtype=BF, enabled=dtype == torch.float32):
        logits, loss = m(ids, labels=ids)
        want = F.cross_entropy(logits[:, :-1].flatten(0, 1), ids[:, 1:].flatten())
    assert type(loss.grad_fn).__name__ == "_NextTokenLossBackward"
    assert loss.dtype == want.dtype
    got = torch.autograd.grad(loss, m.lm_head.weight, retain_graph=True)[0]
    ref = torch.autograd.grad(want, m.lm_head.weight)[0]
    # bf16: the stock gradient exponentiates bf16 log-probabilities (an error
    # of 2^-9 of their size, about 7 here)
    assert (got.float() - ref.float()).norm() <= (3e-2 if dtype == BF else 1e-2) * ref.float().norm()


def _stock_head(h, norm_w, w, eps):
    inv = torch.rsqrt((h * h).mean(-1, keepdim=True) + eps)
    return (h * inv * norm_w) @ w.t()


@pytest.mark.parametrize("tokens,d,vocab", [(2, 8, 8), (3, 72, 1000), (70, 512, 16384), (65, 256, 16392),
                                            (257, 520, 32000), (2100, 4096, 64)])
@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_lm_head(tokens, d, vocab, dtype):
    g = torch.Generator(device="cuda").manual_seed(tokens + d)
    h = torch.randn(1, tokens, d, generator=g, device="cuda").to(dtype).requires_grad_()
    w = (torch.randn(vocab, d, generator=g, device="cuda") / d ** 0.5).to(dtype).requires_grad_()
    norm = RMSNorm(d).to("cuda", dtype)
    with torch.no_grad():
        norm.weight.add_(0.1 * torch.randn(d, generator=g, device="cuda").to(dtype))
    dy = torch.randn(1, tokens, vocab, generator=g, device="cuda").to(BF)
    with torch.autocast("cuda", dtype=BF, enabled=dtype == torch.float32):
        assert lm_head_ok(h, norm, RMSNorm, None, w)
        y = lm_head(h, norm, w)
    got = [y, *torch.autograd.grad(y, (h, norm.weight, w), dy)]
    leaf = [t.detach().to(F64).requires_grad_() for t in (h, norm.weight, w)]
    yd = _stock_head(*leaf, norm.eps)
    want = [yd, *torch.autograd.grad(yd, leaf, dy.to(F64))]
    assert [t.dtype for t in got] == [BF, dtype, dtype, dtype]
    for a, b in zip(got, want):
        # bf16 operands of every product (up to two roundings of 2^-9 each way)
        # and of its result; their errors are independent
        assert (a.to(F64) - b).norm() <= 4 * 2.0 ** -9 * b.norm(), (a.shape, ((a.to(F64) - b).norm() / b.norm()).item())


@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_lm_head_second_derivative_and_frozen_weights(dtype):
    h = torch.randn(1, 5, 64, device="cuda").to(dtype).requires_grad_()
    w = torch.randn(128, 64, device="cuda").to(dtype).requires_grad_()
    norm = RMSNorm(64).to("cuda", dtype)

    def grads(f, *to):
        with torch.autocast("cuda", dtype=BF, enabled=dtype == torch.float32):
            y = f()
        return torch.autograd.grad(y.float().sin().sum(), to, create_graph=True)

    def penalty(f):
        return torch.autograd.grad(grads(f, h)[0].float().square().sum(), (h, w))

    # the same operators, gradients added in another order (bf16 sums)
    for a, b in zip(penalty(lambda: lm_head(h, norm, w)), penalty(lambda: F.linear(norm(h), w))):
        assert a.abs().max() > 0 and (a.float() - b.float()).norm() <= 2e-2 * b.float().norm()
    norm.weight.requires_grad_(False)
    w.requires_grad_(False)
    with torch.autocast("cuda", dtype=BF, enabled=dtype == torch.float32):
        y = lm_head(h, norm, w)
    y.sum().backward()
    assert h.grad.abs().max() > 0 and w.grad is None and norm.weight.grad is None


@pytest.mark.parametrize("tokens,d,vocab", [(5, 64, 128), (4, 512, 16384)])
@pytest.mark.parametrize("rows", [True, False])
def test_lm_head_expanded_gradient(tokens, d, vocab, rows):
    """A sum over the tokens (or over everything) sends an expanded gradient
    back, rows 0 elements apart: the gradients of its contiguous copy."""
    h = torch.randn(1, tokens, d, device="cuda").to(BF).requires_grad_()
    w = torch.randn(vocab, d, device="cuda").to(BF).requires_grad_()
    norm = RMSNorm(d).to("cuda", BF)
    dy = torch.randn(vocab if rows else 1, device="cuda").to(BF).expand(1, tokens, vocab)
    assert dy.stride(1) == 0
    y = lm_head(h, norm, w)
    got = torch.autograd.grad(y, (h, norm.weight, w), dy, retain_graph=True)
    want = torch.autograd.grad(y, (h, norm.weight, w), dy.contiguous())
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("tied", [True, False])
def test_model_uses_lm_head(tied):
    torch.manual_seed(2)
    cfg = MoCConfig(hidden_size=128, intermediate_size=344, num_hidden_layers=1, num_attention_heads=2,
                    vocab_size=1000, max_seq_len=64, tie_word_embeddings=tied)
    m = build_model(cfg, "moc").to("cuda", BF)
    ids = torch.randint(0, 1000, (2, 33), device="cuda")
    assert type(m(ids).grad_fn).__name__ == "_LMHeadBackward"
    seen = []
    hook = m.norm.register_forward_hook(lambda *a: seen.append(1))
    m(ids)
    hook.remove()
    assert seen == [1]


@pytest.mark.parametrize("dtype", [BF, torch.float32])
def test_logits_take_writes_in_place(dtype):
    """Masking or scaling the logits in place, with gradients on: F.linear's result allows it."""
    torch.manual_seed(4)
    cfg = MoCConfig(hidden_size=128, intermediate_size=344, num_hidden_layers=1, num_attention_heads=2,
                    vocab_size=1000, max_seq_len=64)
    m = build_model(cfg, "moc").to("cuda", dtype)
    ids = torch.randint(0, 1000, (2, 9), device="cuda")
    with torch.autocast("cuda", dtype=BF, enabled=dtype == torch.float32):
        got, want = m(ids), m(ids).clone()
        assert type(got.grad_fn).__name__ == "_LMHeadBackward"
        for y in (got, want):
            y[..., 7] = -1.0
            y.div_(2.0)
    grads = [torch.autograd.grad(y, m.lm_head.weight, torch.ones_like(y))[0] for y in (got, want)]
    assert torch.equal(got, want) and torch.equal(*grads)
    assert (grads[0][7] == 0).all()


@pytest.mark.parametrize("tokens,d,vocab", [(70000, 512, 16384), (70000, 512, 32000)])
def test_lm_head_gradients_of_more_than_2_gib_of_logits(tokens, d, vocab):
    g = torch.Generator(device="cuda").manual_seed(8)
    h = torch.randn(1, tokens, d, generator=g, device="cuda").to(BF).requires_grad_()
    w = (torch.randn(vocab, d, generator=g, device="cuda") / d ** 0.5).to(BF).requires_grad_()
    norm = RMSNorm(d).to("cuda", BF)
    dy = torch.randn(1, tokens, vocab, generator=g, device="cuda", dtype=BF)
    got = torch.autograd.grad(lm_head(h, norm, w), (h, norm.weight, w), dy)
    half = [torch.autograd.grad(lm_head(h[:, s], norm, w), (h, norm.weight, w), dy[:, s])
            for s in (slice(0, 35000), slice(35000, None))]
    for a, b, c in zip(got, *half):  # the halves' weight gradients are rounded, and their sum, which a's is not
        assert (a.float() - (b.float() + c.float())).norm() <= 3 * 2.0 ** -9 * a.float().norm()


def test_entry_without_a_copy():
    """moc_next_token_loss_forward: the same loss and row values as with the copy, which is the logits."""
    from moc_amd import _native as N
    x = torch.randn(2, 5, 4104, device="cuda").to(BF)
    labels = torch.randint(0, 4104, (2, 5), device="cuda")
    labels[1, 3] = -100
    keep, bufs, losses = torch.zeros_like(x), torch.zeros(2, 21, device="cuda"), torch.zeros(2, device="cuda")
    for i, name in enumerate(("moc_next_token_loss_forward", "moc_next_token_loss_forward_keep")):
        p = bufs[i].data_ptr()
        N.call(name, x.data_ptr(), 4104, 2, 5, 4104, labels.data_ptr(), -100, p, p + 40, losses[i].data_ptr(),
               N.MOC_F32, p + 80, *((keep.data_ptr(), 4104) if i else ()), N.stream_of(x))
    assert torch.equal(bufs[0], bufs[1]) and torch.equal(losses[0], losses[1]) and torch.equal(keep, x)
