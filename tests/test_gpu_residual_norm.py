"""The leaky residual with its layer norm (bcm_residual_norm_fwd / _bwd)
against float64.

With u = 2^-24, x = v', r = max|x| / std of the row and s = log2(D) + 8 roundings
on any path through a row's sums (lane tree, then one product each):
|err h| <= u s (r + |x^|) |gamma| + 2 u |h|, and each of the three terms of the
row's gradient within u s (1 + r) of its size. Column sums go through at most
300 additions (rows of a thread, 32 row groups, workgroups / 64, 64)."""
import math

import pytest
import torch

from bc_mamba_amd import residual_norm as rn

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _case(dev, rows, D, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    norm = torch.nn.LayerNorm(D)
    with torch.no_grad():
        norm.weight.copy_(r(D))
        norm.bias.copy_(r(D))
    return norm.to(dev), (2.0 * r(rows, D) + 0.5).to(dev), r(rows, D).to(dev), r(rows, D).to(dev), r(rows, D).to(dev)


# every row form at its edges; one row, a ragged last workgroup, rows past one pass of the backward's grid
@pytest.mark.parametrize("rows,D", [(1, 4), (37, 32), (70, 36), (19, 64), (33, 100), (300, 128), (5, 132), (51, 256),
                                    (9001, 256), (40001, 32), (7, 260), (11, 512), (3, 516), (130, 1024)])
@pytest.mark.parametrize("residual", [True, False])
def test_residual_norm(cuda_device, rows, D, residual):
    print(f"residual_norm {rows} {D} {residual}", flush=True)
    norm, v, dv, gh, gv = _case(cuda_device, rows, D, rows + D)
    v, dv = v.requires_grad_(True), dv.requires_grad_(True)
    assert rn._kernel_ok(norm, v, dv)
    if residual:
        h, x = rn.residual_norm(norm, v, dv, 0.95)
        assert torch.equal(x, 0.95 * v + dv) and "ResidualNorm" in type(h.grad_fn).__name__
    else:
        h, x = rn.layer_norm(norm, dv), dv
    x64, w, b = x.detach().double(), norm.weight.detach().double(), norm.bias.detach().double()
    mu, std = x64.mean(1, keepdim=True), (x64.var(1, unbiased=False, keepdim=True) + norm.eps).sqrt()
    xh = (x64 - mu) / std
    s, r = math.log2(D) + 8, x64.abs().amax(1, keepdim=True) / std
    want = xh * w + b
    assert bool(((h.double() - want).abs() <= U * s * (r + xh.abs()) * w.abs() + 2 * U * want.abs() + U * b.abs()).all())
    for use_gv in ([True, False] if residual else [False]):
        leaves = [dv, norm.weight, norm.bias] + ([v] if residual else [])
        got = torch.autograd.grad([h, x] if use_gv else [h], leaves, [gh, gv] if use_gv else [gh], retain_graph=True)
        g = gh.double()
        gw = g * w
        t = (gw, gw.mean(1, keepdim=True), xh * (gw * xh).mean(1, keepdim=True))
        size = gw.abs() + gw.abs().mean(1, keepdim=True) + xh.abs() * (gw * xh).abs().mean(1, keepdim=True)
        dx = (t[0] - t[1] - t[2]) / std + (gv.double() if use_gv else 0.0)
        lim = U * s * (1 + r) * size / std + 2 * U * dx.abs()
        assert bool(((got[0].double() - dx).abs() <= lim).all())
        if residual:
            assert torch.equal(got[3], 0.95 * got[0])
        for c, terms in ((got[1], g * xh), (got[2], g)):
            lim = U * ((300 + s) * terms.abs() + s * r * g.abs()).sum(0)
            assert bool(((c.double() - terms.sum(0)).abs() <= lim).all())


def test_residual_norm_leaves_other_calls_to_torch(cuda_device):
    norm, v, dv, gh, _ = _case(cuda_device, 6, 32, 1)
    ok = rn._kernel_ok
    assert ok(norm, v, dv) and not ok(norm, v, dv.half()) and not ok(norm, v.t().contiguous().t(), dv)
    assert not ok(torch.nn.LayerNorm(30).to(cuda_device), v[:, :30].contiguous())
    assert not ok(torch.nn.LayerNorm(32, elementwise_affine=False).to(cuda_device), v)
    assert not ok(torch.nn.LayerNorm(32, bias=False).to(cuda_device), v)
    assert not ok(norm, v[:1], dv) and not ok(norm, v[:0])
    assert not ok(norm, torch.randn(193, device=cuda_device)[1:].view(6, 32))  # not 16-byte aligned
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not ok(norm, v)
    got = torch.func.vmap(lambda x: rn.layer_norm(norm, x))(v)
    assert torch.equal(got, torch.func.vmap(norm)(v))
    seen = []
    hook = norm.register_forward_hook(lambda *a: seen.append(1))
    rn.layer_norm(norm, v)
    hook.remove()
    assert seen == [1]
    h, x = rn.residual_norm(norm, v[:1], dv, 0.5)  # broadcast, as before
    assert torch.equal(x, 0.5 * v[:1] + dv) and torch.equal(h, norm(x))


def test_residual_norm_gradients_of_v_alone_and_second(cuda_device):
    norm, v, dv, gh, gv = _case(cuda_device, 5, 12, 2)
    v, dv = v.requires_grad_(True), dv.requires_grad_(True)
    h, x = rn.residual_norm(norm, v, dv, 0.95)
    got = torch.autograd.grad(x, [v, dv], gv, retain_graph=True)
    assert torch.equal(got[0], 0.95 * gv) and torch.equal(got[1], gv)
    first = torch.autograd.grad([h, x], [v, norm.weight], [gh, gv.t().contiguous().t()], create_graph=True)
    second = torch.autograd.grad(sum((f * f).sum() for f in first), [dv, norm.weight])
    n64 = torch.nn.LayerNorm(12).to(cuda_device).double()
    n64.load_state_dict({k: t.double() for k, t in norm.state_dict().items()})
    v6, d6 = (t.detach().double().requires_grad_(True) for t in (v, dv))
    x6 = 0.95 * v6 + d6
    f6 = torch.autograd.grad([n64(x6), x6], [v6, n64.weight], [gh.double(), gv.double()], create_graph=True)
    s6 = torch.autograd.grad(sum((f * f).sum() for f in f6), [d6, n64.weight])
    for o, e in zip((*first, *second), (*f6, *s6)):
        assert torch.allclose(o.double(), e, rtol=1e-4, atol=1e-5 * float(e.detach().abs().max()))
