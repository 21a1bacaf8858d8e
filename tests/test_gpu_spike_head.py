"""The fused spike head (e_model.spike_head: bcm_spike_head_fwd / _bwd)
against its composition projections.linear -> torch.sigmoid ->
SpikeSamplerSurrogate: spikes, bitmask and gradients bit for bit, the bias
gradient (of both) within the roundings of its sum (at most 300 additions on
any path, 2^-24 each)."""
import pytest
import torch

from bc_mamba_amd import e_model, projections

pytestmark = pytest.mark.gpu


def _case(dev, B, L, K, Dm, bias, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(dev)
    return [r(B, L, K).requires_grad_(True), (K ** -0.5 * r(Dm, K)).requires_grad_(True),
            r(Dm).requires_grad_(True) if bias else None], r(B, L, Dm)


# every row form of the backward at its edges, ragged time tiles, one step, rows past one pass of the grid
@pytest.mark.parametrize("B,L,K,Dm", [(1, 1, 8, 4), (2, 63, 16, 32), (2, 65, 5, 36), (3, 130, 32, 100), (1, 64, 32, 128),
                                      (2, 257, 48, 256), (20, 500, 32, 256), (1, 33, 16, 260), (1, 40, 16, 1024)])
@pytest.mark.parametrize("bias", [True, False])
def test_spike_head(cuda_device, B, L, K, Dm, bias):
    print(f"spike head {B} {L} {K} {Dm} {bias}", flush=True)
    leaves, ds = _case(cuda_device, B, L, K, Dm, bias, L + Dm)
    sampler = e_model.SpikeSamplerSurrogate(threshold=0.4)
    s = e_model.spike_head(*leaves, sampler)
    assert "SpikeHead" in type(s.grad_fn).__name__
    ref = sampler(torch.sigmoid(projections.linear(*leaves)))
    assert torch.equal(s, ref)
    nw = (L + 31) // 32
    assert torch.equal(s._bcm_event_bits[0][:, :nw], ref._bcm_event_bits[0][:, :nw])
    ps = [t for t in leaves if t is not None]
    got, want = torch.autograd.grad(s, ps, ds), torch.autograd.grad(ref, ps, ds)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    if bias:
        p = torch.sigmoid(projections.linear(*leaves)).detach()
        terms = (ds * (1 - p) * p).reshape(-1, Dm).double()
        assert bool(((got[2].double() - terms.sum(0)).abs() <= 300 * 2.0 ** -24 * terms.abs().sum(0)).all())


def test_spike_head_leaves_other_calls_to_the_composition(cuda_device):
    leaves, ds = _case(cuda_device, 2, 20, 8, 12, True, 1)
    sampler = e_model.SpikeSamplerSurrogate()
    name = lambda s: type(s.grad_fn).__name__
    assert "SpikeHead" in name(e_model.spike_head(*leaves, sampler))
    odd, _ = _case(cuda_device, 2, 20, 8, 10, True, 2)
    assert "SpikeBits" in name(e_model.spike_head(*odd, sampler))
    assert "SpikeBits" in name(e_model.spike_head(leaves[0].half(), leaves[1].half(), leaves[2].half(), sampler))
    assert "SpikeHead" not in name(e_model.spike_head(*leaves, e_model.SpikeSamplerSurrogate(fused_bits=False)))
    assert "SpikeHead" not in name(e_model.spike_head(*leaves, e_model.SpikeSamplerSurrogate(mode="prob")))
    sampler.register_forward_hook(lambda m, a, out: out * 2)
    assert float(e_model.spike_head(*leaves, sampler).detach().amax()) > 1.5
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert e_model.spike_head(*leaves, e_model.SpikeSamplerSurrogate()).dtype == torch.bfloat16


def test_spike_head_second_derivative(cuda_device):
    leaves, ds = _case(cuda_device, 2, 9, 8, 12, True, 3)

    def second(s, ps, d):
        first = torch.autograd.grad(s, ps, d, create_graph=True)
        return torch.autograd.grad(sum((f * f).sum() for f in first), ps)

    got = second(e_model.spike_head(*leaves, e_model.SpikeSamplerSurrogate()), leaves, ds)
    l64 = [t.detach().double().requires_grad_(True) for t in leaves]
    want = second(torch.sigmoid(torch.nn.functional.linear(*l64)), l64, ds.double())
    for o, e in zip(got, want):
        assert torch.allclose(o.double(), e, rtol=1e-4, atol=1e-5 * float(e.abs().max()))
