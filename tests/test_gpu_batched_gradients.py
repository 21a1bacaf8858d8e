"""Several gradients at once (torch.autograd.grad(..., is_grads_batched=True)
and vmap over a backward) through the functions whose backward is a kernel: a
batched gradient is a torch.Tensor by type but has no memory of its own, so
its products are torch's.

Compared with the float64 gradients one by one: the sums have at most 24
terms, each result a few of them in a row, so 100 roundings of 2^-24 of the
largest bound the error (6e-6)."""
import pytest
import torch
import torch.nn.functional as F

from bc_mamba_amd import e_model, projections, residual_norm

pytestmark = pytest.mark.gpu


def _leaves(dev, shapes, dtype=torch.float32):
    g = torch.Generator().manual_seed(5)
    return [torch.randn(*s, generator=g).to(dev, dtype).requires_grad_(True) for s in shapes]


def _norm(cls_dtype, dev):
    return torch.nn.LayerNorm(12).to(dev, cls_dtype)


CASES = {
    "linear": ([(2, 9, 8), (12, 8), (12,)], lambda x, w, b: projections.linear(x, w, b), F.linear),
    "proj_tokens_last": ([(12, 8), (18, 8)], projections.proj_tokens_last, lambda w, h: w @ h.t()),
    "spike_head": ([(2, 9, 8), (12, 8), (12,)],
                   lambda x, w, b: e_model.spike_head(x, w, b, e_model.SpikeSamplerSurrogate()),
                   lambda x, w, b: torch.sigmoid(F.linear(x, w, b))),  # the spikes' gradient is the identity
    "residual_norm": ([(2, 9, 12), (2, 9, 12)],
                      lambda v, dv: residual_norm.residual_norm(_norm(v.dtype, v.device), v, dv, 0.75)[0],
                      lambda v, dv: F.layer_norm(0.75 * v + dv, (12,))),
    "layer_norm": ([(2, 9, 12)], lambda x: residual_norm.layer_norm(_norm(x.dtype, x.device), x),
                   lambda x: F.layer_norm(x, (12,))),
}


@pytest.mark.parametrize("name", list(CASES))
def test_batched_gradients(cuda_device, name):
    print(f"batched gradients {name}", flush=True)
    shapes, fn, ref = CASES[name]
    ps = _leaves(cuda_device, shapes)
    out = fn(*ps)
    gs = torch.randn(3, *out.shape, generator=torch.Generator().manual_seed(6)).to(cuda_device)
    p64 = _leaves(cuda_device, shapes, torch.float64)
    o64 = ref(*p64)
    want = [torch.stack(t) for t in zip(*(torch.autograd.grad(o64, p64, g.double(), retain_graph=True) for g in gs))]
    at_once = torch.autograd.grad(out, ps, gs, is_grads_batched=True, retain_graph=True)
    mapped = torch.func.vmap(lambda g: torch.autograd.grad(out, ps, g, retain_graph=True))(gs)
    for got in (at_once, mapped):
        for a, b in zip(got, want):
            assert float((a.double() - b).abs().max()) <= 100 * 2.0 ** -24 * max(1.0, float(b.abs().max()))
