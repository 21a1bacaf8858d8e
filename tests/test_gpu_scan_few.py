"""The depthwise forward scan of few channels (a workgroup a channel, the
states over its waves) against the recurrence event by event in float64:
g_s <- a_s g_s + dt u^2, y = D u + u sum_s g_s W_B W_C.

Every term of g is positive, so a bound follows the recurrence: with u = 2^-24
a step rounds g within 8 u (decay from exp2 of a rounded exponent, product,
sum), e <- a (e + 8 u g) + 8 u dt u^2, and the lane scan and the sum over states
add 64 u of g."""
import pytest
import torch

from bc_mamba_amd import selective_scan_cuda as sc

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _problem(dev, NC, D, N, longest, dtype, long_gap, positive_a, seed):
    g = torch.Generator().manual_seed(seed)
    lens = torch.randint(0, longest + 1, (NC,), generator=g)
    lens[:3] = torch.tensor([longest, 0, 1])
    cu = torch.zeros(NC + 1, dtype=torch.int32)
    cu[1:] = lens.cumsum(0)
    E = int(cu[-1])
    k = torch.randint(1, 12, (E,), generator=g, dtype=torch.int32)
    if long_gap:
        k[::97] = 300  # past the decay table
    r = lambda *s: torch.rand(*s, generator=g)
    A = -(0.2 + 2.0 * r(D, N))
    if positive_a:
        A[0, 0] = 0.01  # the decays are multiplied out
    p = (k, cu, 0.02 * r(D), 0.01 + 0.1 * r(D), A, torch.randn(D, N, generator=g), torch.randn(D, N, generator=g),
         torch.randn(D, generator=g))
    u, z = torch.randn(E, generator=g).to(dtype), torch.randn(E, generator=g).to(dtype)
    return [t.to(dev) for t in (u, z, *p)], lens.to(dev)


def _reference(u, k, cu, lens, dti, dta, A, WB, WC, Dp, pass_len):
    """y, sum, bound of its error, and {event count: (g W_B, bound)} at every
    pass start."""
    NC, D = lens.numel(), A.size(0)
    d = torch.arange(NC, device=u.device) % D
    y, acc, lim = (torch.zeros(u.numel(), dtype=torch.float64, device=u.device) for _ in range(3))
    u, dti, dta, A, WB, WC, Dp = (t.double() for t in (u, dti, dta, A, WB, WC, Dp))
    gs = torch.zeros(NC, A.size(1), dtype=torch.float64, device=u.device)
    e, starts = torch.zeros_like(gs), {}
    for t in range(int(lens.max())):
        if t and t % pass_len == 0:
            starts[t // pass_len] = (gs * WB[d], (e + 64 * U * gs) * WB[d].abs())
        c = (lens > t).nonzero().squeeze(1)
        i, dc = cu[c].long() + t, d[c]
        dt = dti[dc] * (k[i] - 1) + dta[dc]
        a, x = torch.exp(dt[:, None] * A[dc]), (dt * u[i] ** 2)[:, None]
        e[c] = a * (e[c] + 8 * U * gs[c]) + 8 * U * x
        gs[c] = a * gs[c] + x
        w = WB[dc] * WC[dc]
        acc[i] = (gs[c] * w).sum(1)
        lim[i] = ((e[c] + 64 * U * gs[c]) * w.abs()).sum(1)
        y[i] = Dp[dc] * u[i] + u[i] * acc[i]
    return y, acc, lim, starts


# waves a channel follow the states (8, 4, 2), items a lane the longest channel
@pytest.mark.parametrize("NC,D,N,longest,dtype,z,gap,pos", [
    (5, 5, 16, 256, torch.float32, False, False, False), (9, 4, 9, 257, torch.float32, True, False, False),
    (512, 128, 16, 512, torch.float32, False, True, False), (700, 700, 5, 513, torch.bfloat16, True, False, False),
    (1030, 515, 16, 300, torch.float16, False, False, True), (1000, 500, 2, 200, torch.float32, False, False, False),
    (12, 6, 64, 1024, torch.float32, False, True, False), (8, 8, 16, 1025, torch.bfloat16, False, False, False),
    (6, 3, 33, 2600, torch.float32, True, False, True), (4, 2, 16, 4500, torch.float32, False, True, False)])
def test_scan_few_channels(cuda_device, NC, D, N, longest, dtype, z, gap, pos):
    print(f"scan few {NC} {D} {N} {longest} {dtype} {z} {gap} {pos}", flush=True)
    (u, zt, k, cu, *params), lens = _problem(cuda_device, NC, D, N, longest, dtype, gap, pos, NC + N)
    A = params[2]
    chunk_g = sc.chunk_states_buffer(u, cu, longest, A)
    acc = torch.zeros(u.numel(), dtype=torch.float32, device=u.device)
    res = sc.fwd_flat_ch(u, k, cu, longest, *params, zt if z else None, is_depthwise_bc=True, _chunk_g=chunk_g,
                         _acc=acc)
    pass_len = chunk_g.bcm_pass_len if chunk_g is not None else 2048
    y, want, lim, starts = _reference(u, k, cu, lens, *params, pass_len)
    assert bool(((acc.double() - want).abs() <= lim).all())
    rnd = {torch.float32: U, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    uo = u.double().abs()
    ylim = uo * lim + 2 * U * (uo * want.abs() + y.abs()) + 4 * U * uo * params[5].double().abs().max()
    assert bool(((res[0].double() - y).abs() <= ylim + rnd * y.abs() + 1e-7 * (rnd > U)).all())
    if z:
        yz = y * zt.double() * torch.sigmoid(zt.double())
        assert bool(((res[2].double() - yz).abs() <= ylim * zt.double().abs() + (rnd + 16 * U) * yz.abs()
                     + 1e-7 * (rnd > U)).all())
    for row, (s, sl) in starts.items():
        live = lens > row * pass_len
        if chunk_g is not None:
            assert bool(((chunk_g[:, row].double() - s).abs() <= sl)[live].all())
        if row * pass_len % 2048 == 0:
            x = res[1].view(NC, -1, 2 * N)[:, row * pass_len // 2048 - 1, 1::2]
            assert bool(((x.double() - s).abs() <= sl)[lens >= row * pass_len].all())
    x = res[1].view(NC, -1, 2 * N)
    ended = (lens[:, None] + 2047) // 2048 <= torch.arange(x.size(1), device=x.device)
    assert bool((x[ended] == 0).all())
