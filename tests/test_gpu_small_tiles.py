"""The small-tile GEMM launches (products whose 256x256 tiles would leave most
CUs idle) against 64-bit products, at tile edges and K remainders."""
import pytest
import torch

from moc_amd import kernels as K

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _mat(rows, cols, gen, contiguous_along_cols=True):
    """[rows, cols] bf16 with 16-byte aligned rows of the chosen orientation;
    the pad columns hold NaN (never to be read as data)."""
    r, c = (rows, cols) if contiguous_along_cols else (cols, rows)
    buf = torch.full((r, K.row_pitch(c, BF)), float("nan"), dtype=BF, device="cuda")
    buf[:, :c] = torch.randn(r, c, generator=gen, device="cuda").to(BF)
    t = buf[:, :c]
    return t if contiguous_along_cols else t.t()


def _check(out, ref, mags, k):
    """out within the bf16 rounding of a sum whose f32 accumulation is off by
    at most k 2^-24 of the sum of magnitudes (f32 outputs: the latter alone)."""
    eps = 2.0 ** -8 if out.dtype == BF else 0.0
    bound = eps * ref.abs() + (1 + eps) * (k + 2) * 2.0 ** -24 * mags + 1e-30
    bad = (out.double() - ref).abs() > bound
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} off, worst " \
                          f"{((out.double() - ref).abs() / bound).max().item():.3g} of the bound"


SHAPES = [
    # M, N, K: one tile; tile edges; K remainders of 1 to 7 and of whole
    # chunks; long K (split); the largest products the rule gives small tiles
    (17, 64, 64), (64, 65, 72), (65, 129, 130), (129, 127, 1000), (200, 1000, 517), (1, 8, 8),
    (48, 2048, 5461), (333, 300, 4097), (1000, 1024, 2736), (1024, 2736, 1000), (2048, 2048, 5456),
    # 70 and 49 tiles of 256 with a long K: back on three and five K parts
    (1280, 3398, 5000), (1619, 1728, 7546),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("a_kc", [True, False])
@pytest.mark.parametrize("b_kc", [True, False])
def test_layouts_and_edges(m, n, k, a_kc, b_kc):
    gen = torch.Generator(device="cuda").manual_seed(m * 7 + n * 3 + k)
    a = _mat(m, k, gen, a_kc)
    b = _mat(k, n, gen, not b_kc)
    ref = a.double() @ b.double()
    mags = a.double().abs() @ b.double().abs()
    _check(K.gemm(a, b), ref, mags, k)
    _check(K.gemm(a, b, out_dtype=torch.float32), ref, mags, k)


@pytest.mark.parametrize("m,n,k", [(64, 128, 256), (100, 512, 1376), (1000, 1024, 2736), (300, 513, 333)])
def test_two_products_and_residual(m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, a2 = _mat(m, k, gen), _mat(m, k + 40, gen)
    b, b2 = _mat(k, n, gen), _mat(k + 40, n, gen)
    ref = a.double() @ b.double() + a2.double() @ b2.double()
    mags = a.double().abs() @ b.double().abs() + a2.double().abs() @ b2.double().abs()
    _check(K.gemm(a, b, a2=a2, b2=b2), ref, mags, 2 * k + 40)
    res = _mat(m, n, gen)
    out = K.gemm(a, b, residual=res)
    plain = K.gemm(a, b)  # the same sums, rounded to bf16 before the residual is added
    assert torch.equal(out, (plain.float() + res.float()).to(BF))


@pytest.mark.parametrize("m", [2, 17, 64, 65, 200, 512, 1000])
@pytest.mark.parametrize("n1,n2,k", [(512, 512, 256), (1376, 1000, 520), (5461, 5461, 2048)])
def test_pair(m, n1, n2, k):
    gen = torch.Generator(device="cuda").manual_seed(m + n1 + k)
    x, w1, w2 = _mat(m, k, gen), _mat(n1, k, gen), _mat(n2, k, gen)
    o1, o2 = K.linear_pair(x, w1, w2, out1=K.padded_empty(m, n1, BF, "cuda"),
                           out2=K.padded_empty(m, n2, BF, "cuda"))
    for o, w in ((o1, w1), (o2, w2)):
        _check(o, x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t(), k)


def test_without_workspace():
    """A long-K product whose caller passes no workspace runs unsplit."""
    from moc_amd import _native as N
    gen = torch.Generator(device="cuda").manual_seed(5)
    m, n, k = 48, 512, 4096
    a, b = _mat(m, k, gen), _mat(k, n, gen)
    out = torch.empty(m, n, dtype=BF, device="cuda")
    N.call("moc_gemm_ws", N.MOC_BF16, m, n, k, a.data_ptr(), a.stride(0), 1, b.data_ptr(), b.stride(0), 1, 0,
           None, 0, 0, None, 0, 0, out.data_ptr(), n, N.MOC_BF16, None, 0, N.stream_of(a))
    _check(out, a.double() @ b.double(), a.double().abs() @ b.double().abs(), k)


@pytest.mark.parametrize("m,n,k", [(7086, 704, 1699), (2048, 2560, 520), (9216, 328, 1376), (3346, 1216, 2824),
                                   (3604, 712, 5544)])
@pytest.mark.parametrize("b_kc", [True, False])
def test_plans_on_either_side_of_the_small_tiles_line(m, n, k, b_kc):
    """128-row tiles, small tiles, 128-row tiles in two parts, a K split."""
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, b = _mat(m, k, gen), _mat(k, n, gen, not b_kc)
    ref, mags = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    _check(K.gemm(a, b), ref, mags, k)
    res = _mat(m, n, gen)
    assert torch.equal(K.gemm(a, b, residual=res), (K.gemm(a, b).float() + res.float()).to(BF))
