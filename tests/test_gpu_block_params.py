"""The block's scan parameters from one kernel each way against the torch
form in float64: both softplus branches, missing gradients."""
import pytest
import torch
import torch.nn.functional as F

from bc_mamba_amd import e_model
from conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,N", [(1, 1), (3, 5), (64, 16), (257, 64)])
def test_block_params(cuda_device, D, N):
    g = torch.Generator().manual_seed(D + N)
    a0 = 12.0 * torch.randn(D, generator=g)
    a0[0] = 25.0  # past the softplus threshold
    a1, al, w = 3.0 * torch.randn(D, generator=g), torch.randn(D, N, generator=g), torch.randn(D, 2 * N, generator=g)
    leaves = [t.to(cuda_device).requires_grad_(True) for t in (a0, a1, al, w)]
    out = e_model._BlockParamsFn.apply(*leaves, 1e-6)
    r = [t.double().requires_grad_(True) for t in (a0, a1, al, w)]
    want = (F.softplus(r[0]) + 1e-6, F.softplus(r[1]) + 1e-6, -torch.exp(r[2]), r[3][:, :N], r[3][:, N:])
    for o, e in zip(out, want):
        assert_close(o.detach().cpu(), e.detach(), 2e-6, 2e-7)
    gs = [torch.randn(o.shape, generator=g) for o in want]
    got = torch.autograd.grad(out, leaves, [t.to(cuda_device) for t in gs], retain_graph=True)
    ref = torch.autograd.grad(want, r, [t.double() for t in gs], retain_graph=True)
    for o, e in zip(got, ref):
        assert_close(o.cpu(), e, 2e-6, 2e-7)
    # only A and W_C used
    got = torch.autograd.grad([out[2], out[4]], leaves, [gs[2].to(cuda_device), gs[4].to(cuda_device)])
    ref = torch.autograd.grad([want[2], want[4]], r, [gs[2].double(), gs[4].double()], allow_unused=True)
    for o, e in zip(got, ref):
        assert_close(o.cpu(), torch.zeros_like(o.cpu()) if e is None else e, 2e-6, 2e-7)


def test_block_takes_the_kernel_only_for_its_own_parameters(cuda_device):
    blk = e_model.Mamba(d_model=16, d_state=8, device=cuda_device)
    ours = blk._scan_params()
    assert all(o.grad_fn is ours[0].grad_fn for o in ours)
    blk.delta_gen.levels = lambda: (torch.full((32,), 0.5, device=cuda_device),) * 2  # a level generator of the user's
    assert float(blk._scan_params()[0][0]) == 0.5
    del blk.delta_gen.levels
    ref = (*blk.delta_gen.levels(), -torch.exp(blk.A_log), blk.W_BC[:, :8], blk.W_BC[:, 8:])
    for o, e in zip(ours, ref):
        assert torch.allclose(o, e, rtol=2e-6, atol=0)


def test_block_params_second_derivative(cuda_device):
    g = torch.Generator().manual_seed(1)
    raw = [torch.randn(s, generator=g) for s in ((4,), (4,), (4, 3), (4, 6))]
    leaves = [t.to(cuda_device).requires_grad_(True) for t in raw]
    r = [t.double().requires_grad_(True) for t in raw]

    def second(out, xs):
        first = torch.autograd.grad(sum((o * o).sum() for o in out), xs, create_graph=True)
        return torch.autograd.grad(sum((f * f).sum() for f in first), xs)

    want = second((F.softplus(r[0]) + 1e-6, F.softplus(r[1]) + 1e-6, -torch.exp(r[2]), r[3][:, :3], r[3][:, 3:]), r)
    for o, e in zip(second(e_model._BlockParamsFn.apply(*leaves, 1e-6), leaves), want):
        assert_close(o.cpu(), e, 1e-5, 1e-6)
