"""The per-event B/C scans at every workgroup shape: channels per model
channel around the four of a wave and the 32 of a workgroup, dstates that
leave states unevenly shared or single, passes of 128 events that end in the
middle, the last events of the streams (item-by-item loads at the operands'
end), tile widths inside and outside the 8-event groups. Against the float64
oracle, with the comparison of test_gpu_scan_modes."""
import numpy as np
import pytest
import torch

from test_gpu_scan_modes import _case, _check_fwd_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 3, 16])
@pytest.mark.parametrize("B,L", [(1, 700), (4, 260), (5, 130), (9, 100), (17, 64), (33, 300)])
def test_per_event_shapes(cuda_device, B, L, N):
    print(f"scan var B={B} L={L} N={N}", flush=True)
    c = _case(B, 3, L, 0.5, N, torch.float32, 100 * B + N, with_z=B % 2 == 1, empty_every=4)
    Bt = torch.randn(N, c["E"], generator=c["g"])
    Ct = torch.randn(N, c["E"], generator=c["g"])
    _check_fwd_bwd(c, Bt, Ct, torch.float32, cuda_device)


@pytest.mark.parametrize("T", [1, 8, 12, 2048])
@pytest.mark.parametrize("B", [2, 20])
def test_tiled_shapes(cuda_device, B, T):
    print(f"scan var tiled B={B} T={T}", flush=True)
    c = _case(B, 3, 400, 0.4, 6, torch.float32, 7 * B + T, with_z=True)
    tiles = (np.diff(c["cu"]) + T - 1) // T
    toff = np.concatenate([[0], np.cumsum(tiles)])[:-1]
    nt = int(tiles.sum())
    Bt = torch.randn(nt, 6, T, generator=c["g"])
    Ct = torch.randn(nt, 6, T, generator=c["g"])
    _check_fwd_bwd(c, Bt, Ct, torch.float32, cuda_device, tile_offsets=toff, T=T)


def test_two_runs_are_bit_equal(cuda_device):
    c = _case(6, 5, 900, 0.4, 16, torch.float32, 3, with_z=True)
    Bt = torch.randn(16, c["E"], generator=c["g"])
    Ct = torch.randn(16, c["E"], generator=c["g"])
    r1, g1 = _check_fwd_bwd(c, Bt, Ct, torch.float32, cuda_device)
    r2, g2 = _check_fwd_bwd(c, Bt, Ct, torch.float32, cuda_device)
    assert all(torch.equal(a, b) for a, b in zip(list(r1) + list(g1), list(r2) + list(g2)))
