"""Captured products of solvers whose spectral kernel takes more than 64 KB of
LDS (113 to 128 levels in mixed precision) and of their neighbours: every
replay, with eager work and position updates in between, gives the eager
product's bits."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

ETA = 1 / (6 * np.pi)


@pytest.mark.parametrize("precision,nz", [("mixed", 112), ("mixed", 113), ("mixed", 128), ("mixed", 129),
                                          ("double", 128)])
def test_replays_give_the_eager_bits(precision, nz):
    import torch
    from doublyperiodicstokes_amd import DPStokes, StokesParameters
    say("captured product, %s, %d levels" % (precision, nz))
    nx, N, Lz = 48, 150, 0.33 * nz
    L = 0.5 * nx
    par = StokesParameters(viscosity=ETA, Lx=L, Ly=L, zmin=0.0, zmax=Lz, w=6, w_d=6, beta=1.785 * 6,
                           beta_d=1.785 * 6, nx=nx, ny=nx, nz=nz, mode="slit", precision=precision)
    dt = torch.float64 if precision == "double" else torch.float32
    rng = np.random.RandomState(nz)
    dev = lambda a: torch.tensor(a, dtype=dt, device="cuda")  # noqa: E731
    pos = [dev(np.stack([rng.uniform(0, L, N), rng.uniform(0, L, N), rng.uniform(0.5, Lz - 0.5, N)], 1).ravel())
           for _ in range(3)]
    F, T = dev(rng.normal(size=3 * N)), dev(rng.normal(size=3 * N))
    s = DPStokes()
    s.initialize(par, N)
    s.setPositions(pos[0])
    want = []
    for p in pos:
        s.setPositions(p)
        want.append([a.cpu().numpy() for a in s.mdot_device(F, T)])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = s.mdot_device(F, T)
    for i in (0, 1, 2, 1, 0):
        s.setPositions(pos[i])
        g.replay()
        torch.cuda.synchronize()
        assert all(np.array_equal(a.cpu().numpy(), b) for a, b in zip(out, want[i]))
        _ = (F * 2.0).sum().item()
        assert all(np.array_equal(a.cpu().numpy(), b) for a, b in zip(s.mdot_device(F, T), want[i]))
    s.clear()
