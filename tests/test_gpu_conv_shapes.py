"""The dense causal convolution where its workgroup shapes change: rows of a
few steps (many to a workgroup), rows of one step more or less than the
threads cover, rows of several workgroups, odd lengths (vectors at any element
alignment), storage that starts between 16-byte boundaries, widths whose halo
reaches past both ends of a row. Against float64."""
import pytest
import torch

from bc_mamba_amd.causal_conv1d import causal_conv1d_fn
from conftest import assert_close

pytestmark = pytest.mark.gpu

TOL = {torch.float32: (1e-5, 1e-6), torch.bfloat16: (1.6e-2, 1e-3), torch.float16: (2e-3, 2e-4)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,L,K", [(1, 1, 1, 4), (3, 5, 3, 8), (70, 2, 9, 4), (2, 33, 64, 2), (3, 7, 255, 4),
                                     (2, 3, 2047, 4), (2, 3, 2049, 8), (1, 2, 5001, 4), (9, 40, 130, 3)])
def test_conv_shapes(cuda_device, B, D, L, K, dtype):
    print(f"conv {B} {D} {L} {K} {dtype}", flush=True)
    g = torch.Generator().manual_seed(B + D + L + K)
    # storage that starts one element into an allocation
    x = torch.randn(B * D * L + 1, generator=g).to(dtype).to(cuda_device)[1:].view(B, D, L).requires_grad_(True)
    w = torch.randn(D, K, generator=g).to(cuda_device).requires_grad_(True)
    b = torch.randn(D, generator=g).to(cuda_device).requires_grad_(True)
    dout = torch.randn(B, D, L, generator=g).to(dtype).to(cuda_device)
    out = causal_conv1d_fn(x, w, b, activation="silu")
    grads = torch.autograd.grad(out, [x, w, b], dout)
    r = [t.detach().double().requires_grad_(True) for t in (x, w, b)]
    pad = torch.nn.functional.pad(r[0], (K - 1, 0))
    pre = r[2][:, None] + sum(r[1][:, k, None] * pad[..., k:k + L] for k in range(K))
    ref = pre * torch.sigmoid(pre)
    want = torch.autograd.grad(ref, r, dout.double())
    rtol, atol = TOL[dtype]
    for name, a, e in zip(("out", "dx"), (out, grads[0]), (ref, want[0])):
        assert_close(a.detach().float().cpu(), e.detach().cpu(), rtol, atol, name)
    # dw, db: fp32 sums of B L terms, each within 8 roundings of fp32
    n = B * L
    for name, a, e in zip(("dw", "db"), grads[1:], want[1:]):
        assert_close(a.cpu(), e.cpu(), 1e-5, (8 + n ** 0.5) * 2.0 ** -23 * 4, name)
