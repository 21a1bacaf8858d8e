"""GPU parity of the fp32 product on the fp16 matrix cores (bcm_gemm_f32,
projections.mm) against float64.

Bound of one result, with S = sum over k of |a||b|: each operand value is
represented within 2^-23 of itself or 2^-34 of its row's largest, the dropped
lo lo product is within 2^-22, and the fp32 sum rounds three times per 16
products, once per slice and once at the end, each rounding within 2^-23 of
S (the matrix cores may truncate):
|err| <= (2^-21 + (3 K / 16 + 70) 2^-23) S + 2^-33 (max|a| sum|b| + max|b| sum|a|)."""
import pytest
import torch

from bc_mamba_amd import _native as nat
from bc_mamba_amd import projections as pj

pytestmark = pytest.mark.gpu


def _bound(a, b):
    """a [M, K], b [K, N] float64."""
    K = a.size(1)
    s = a.abs() @ b.abs()
    tail = a.abs().amax(1, keepdim=True) * b.abs().sum(0) + a.abs().sum(1, keepdim=True) * b.abs().amax(0)
    return (2.0 ** -21 + (3 * K / 16 + 70) * 2.0 ** -23) * s + 2.0 ** -33 * tail


def _check(x, y, bias=None):
    assert pj._kernel_form(x, y, bias) is not None
    got = pj.mm(x, y, bias)
    a, b = x.double(), y.double()
    want = a @ b + (bias.double() if bias is not None else 0.0)
    lim = _bound(a, b) + (2.0 ** -23 * want.abs() if bias is not None else 0.0) + 1e-44
    assert bool(((got.double() - want).abs() <= lim).all()), float(((got.double() - want).abs() / lim).max())
    return got


def _operands(M, N, K, form, dev, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(dev) if form[0] else torch.randn(K, M, generator=g).to(dev).t()
    y = torch.randn(K, N, generator=g).to(dev) if form[1] else torch.randn(N, K, generator=g).to(dev).t()
    return x, y


# tile edges (128), k-chunk edges (32), one element, split sums with a ragged last slice
SIZES = [(1, 1, 1), (127, 129, 31), (128, 128, 32), (129, 127, 33), (300, 3, 65), (64, 200, 96), (131, 66, 515),
         (256, 128, 4096), (40, 48, 20001), (257, 64, 8195)]
# (k-contiguous x, n-contiguous y)
FORMS = [(True, False), (True, True), (False, True)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("M,N,K", SIZES)
def test_gemm_sizes(cuda_device, M, N, K, form):
    print(f"gemm {M} {N} {K} {form}", flush=True)
    x, y = _operands(M, N, K, form, cuda_device, seed=M + N + K)
    _check(x, y)
    _check(x, y, torch.randn(N, generator=torch.Generator().manual_seed(1)).to(cuda_device))


def test_gemm_strided_operands(cuda_device):
    """Leading dimensions above the row length, also odd ones."""
    g = torch.Generator().manual_seed(2)
    wide = torch.randn(200, 333, generator=g).to(cuda_device)
    x, y = wide[:150, 5:70], torch.randn(65, 131, generator=g).to(cuda_device)[:, 2:100]
    _check(x, y)
    _check(wide[7:72, 1:140].t(), y)


@pytest.mark.parametrize("form", FORMS)
def test_gemm_scales_follow_the_rows(cuda_device, form):
    """Rows of very different size, values that grow along k past the first
    chunk's headroom (the scales are lowered on the way), leading zeros, a
    zero row, subnormal values."""
    g = torch.Generator().manual_seed(3)
    K = 700
    a = torch.randn(150, K, generator=g) * torch.exp2(60 * torch.rand(150, 1, generator=g) - 30)
    a = a * torch.exp2(torch.linspace(-40, 30, K))
    a[:40, :300] = 0.0
    a[41] = 0.0
    a[42] *= 1e-38
    b = torch.randn(K, 140, generator=g) * torch.exp2(40 * torch.rand(140, generator=g) - 20)
    b[:, 10] = 0.0
    x = a.to(cuda_device) if form[0] else a.t().contiguous().to(cuda_device).t()
    y = b.to(cuda_device) if form[1] else b.t().contiguous().to(cuda_device).t()
    _check(x, y)


def test_gemm_infinities_and_nan(cuda_device):
    g = torch.Generator().manual_seed(4)
    a, b = torch.randn(200, 300, generator=g), torch.randn(300, 150, generator=g)
    a[3, 7], a[5, 290], b[200, 4], b[7, 8] = float("inf"), float("nan"), -float("inf"), 0.0
    x, y = a.to(cuda_device), b.to(cuda_device)
    got, want = pj.mm(x, y).double(), x.double() @ y.double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fin = want.isfinite()
    assert torch.equal(got.sign()[want.isinf()], want.sign()[want.isinf()])
    a[3, 7] = a[5, 290] = 0.0
    b[200, 4] = 0.0
    lim = _bound(a.double(), b.double()).to(cuda_device)
    assert bool(((got - want).abs()[fin] <= lim[fin]).all())


def test_projection_gradients(cuda_device):
    """linear and proj_tokens_last against float64, and the second derivative
    through linear (which the kernel leaves to torch)."""
    g = torch.Generator().manual_seed(5)
    T, I, O = 8192 + 37, 48, 72
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda_device)
    x, w, b, gy = rnd(T, I), rnd(O, I), rnd(O), rnd(T, O)
    leaves = [t.clone().requires_grad_(True) for t in (x, w, b)]
    y = pj.linear(*leaves)
    grads = torch.autograd.grad(y, leaves, gy)
    for got, a, c in ((y, x, w.t()), (grads[0], gy, w), (grads[1], gy.t(), x)):
        want = a.double() @ c.double() + (b.double() if got is y else 0.0)
        assert bool(((got.double() - want).abs() <= _bound(a.double(), c.double()) + 2.0 ** -23 * want.abs()).all())
    wi, h, gi = rnd(O, I).requires_grad_(True), rnd(T, I).requires_grad_(True), rnd(O, T)
    out = pj.proj_tokens_last(wi, h)
    dw, dh = torch.autograd.grad(out, [wi, h], gi)
    for got, a, c in ((out, wi, h.t()), (dw, gi, h), (dh, gi.t(), wi)):
        a, c = a.detach().double(), c.detach().double()
        assert bool(((got.double() - a @ c).abs() <= _bound(a, c)).all())
    leaves = [t[:64].clone().requires_grad_(True) if t.size(0) == T else t.clone().requires_grad_(True) for t in (x, w, b)]
    (gx,) = torch.autograd.grad(pj.linear(*leaves).pow(2).sum(), leaves[:1], create_graph=True)
    (gw,) = torch.autograd.grad(gx.sum(), leaves[1:2])
    ref = [t.detach().double().requires_grad_(True) for t in leaves]
    (rx,) = torch.autograd.grad(torch.nn.functional.linear(*ref).pow(2).sum(), ref[:1], create_graph=True)
    (rw,) = torch.autograd.grad(rx.sum(), ref[1:2])
    assert torch.allclose(gw.double(), rw, rtol=1e-4, atol=1e-4 * float(rw.abs().max()))


def test_gemm_leaves_other_products_to_torch(cuda_device):
    f = torch.randn(16, 16, device=cuda_device)
    assert pj._kernel_form(f, f) is not None
    assert pj._kernel_form(f.half(), f.half()) is None
    assert pj._kernel_form(f.t(), f.t()) is None  # k-major x with a row-major y
    assert pj._kernel_form(f[:, ::2], f[:8]) is None
    assert pj._kernel_form(f[:1].expand(16, 16), f) is None  # overlapping rows
    assert pj._kernel_form(f.clone().requires_grad_(True), f) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert pj._kernel_form(f, f) is None
    for x, y in ((f.t(), f.t()), (f[:, ::2], f[:8]), (f[:1].expand(16, 16), f)):
        assert torch.allclose(pj.mm(x, y), x @ y)


@pytest.mark.parametrize("form", FORMS)
def test_gemm_errors_do_not_add_up(cuda_device, form):
    """The errors of many results have no common direction: their mean over
    n = 4096 x 256 results stays within 8 / sqrt(n) of their size (a rounding
    in one direction leaves it near a twentieth of it)."""
    x, y = _operands(4096, 256, 256, form, cuda_device, seed=6)
    err = pj.mm(x, y).double() - x.double() @ y.double()
    rms = float(err.pow(2).mean().sqrt())
    assert abs(float(err.mean())) <= 8.0 * rms / (4096 * 256) ** 0.5
    for dim, n in ((0, 4096), (1, 256)):  # and along either side
        assert float(err.sum(dim).pow(2).mean().sqrt()) <= 2.0 * rms * n ** 0.5
