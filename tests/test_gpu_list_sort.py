"""Tile lists at the length where the sort changes form (counting up to 512, a
bit per particle beyond, 131072 particles at a time) and one past it.  Spread
grids against the FP64 oracle (rel-L2 <= 1e-11), and the same bits from every
build of the same positions."""
import numpy as np
import pytest

from oracle.dp_oracle import OracleDPStokes
from test_gpu_parity import TOL64, rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 511, 512, 513, 1025, 8192, 8193, 20000])
def test_crowded_lists(N):
    import torch
    from doublyperiodicstokes_amd import DPStokes, StokesParameters
    say("lists of %d particles" % N)
    h, nx, ny, nz, w, eta, Lz = 0.5, 64, 24, 12, 4, 0.7, 4.0
    par = StokesParameters(viscosity=eta, Lx=h * nx, Ly=h * ny, zmin=0.0, zmax=Lz, w=w, w_d=0, beta=1.785 * w, nx=nx,
                           ny=ny, nz=nz, mode="slit", precision="double")
    rng = np.random.RandomState(N)
    # supports over columns 8 .. 24 and 7 .. 12: every particle in three tiles
    pos = np.stack([rng.uniform(10 * h, 22 * h, N), rng.uniform(9.6 * h, 10.4 * h, N), rng.uniform(0, Lz, N)], 1).ravel()
    F = rng.normal(size=3 * N)
    ref = OracleDPStokes("slit", h * nx, h * ny, 0.0, Lz, nx, ny, nz, eta, w, 1.785 * w)
    ref.set_positions(pos)
    want = ref.spread_forces(F, None)
    s = DPStokes()
    s.initialize(par, N)
    Fd = torch.from_numpy(F)
    first = None
    for _ in range(3):
        s.setPositions(pos)
        got = s.stage_spread(Fd).cpu().numpy()
        first = got if first is None else first
        assert np.array_equal(got, first)
    e = rel_l2(first, want)
    say("  rel-L2 %.3e" % e)
    assert e <= TOL64
    s.clear()


def test_crowded_lists_among_many_particles():
    """One tile's list over more than two windows of particle indices: 6000 of
    270000 particles under the same tiles, the others elsewhere."""
    import torch
    from doublyperiodicstokes_amd import DPStokes, StokesParameters
    say("crowded lists among 270000 particles")
    h, nx, ny, nz, w, eta, Lz, N = 0.5, 256, 128, 6, 4, 0.7, 1.5, 270000
    par = StokesParameters(viscosity=eta, Lx=h * nx, Ly=h * ny, zmin=0.0, zmax=Lz, w=w, w_d=0, beta=1.785 * w, nx=nx,
                           ny=ny, nz=nz, mode="slit", precision="double")
    rng = np.random.RandomState(4)
    pos = np.stack([rng.uniform(40 * h, 250 * h, N), rng.uniform(20 * h, 120 * h, N), rng.uniform(0, Lz, N)], 1)
    crowd = np.concatenate([[0, 131071, 131072, 262143, 262144, N - 1], rng.choice(np.arange(1, N - 1), 6000, False)])
    pos[crowd, 0] = rng.uniform(10 * h, 22 * h, len(crowd))
    pos[crowd, 1] = rng.uniform(9.6 * h, 10.4 * h, len(crowd))
    F = rng.normal(size=3 * N)
    ref = OracleDPStokes("slit", h * nx, h * ny, 0.0, Lz, nx, ny, nz, eta, w, 1.785 * w)
    ref.set_positions(pos.ravel())
    want = ref.spread_forces(F, None)
    s = DPStokes()
    s.initialize(par, N)
    Fd = torch.from_numpy(F)
    s.setPositions(pos.ravel())
    got = s.stage_spread(Fd).cpu().numpy()
    s.setPositions(pos.ravel())
    assert np.array_equal(s.stage_spread(Fd).cpu().numpy(), got)
    e = rel_l2(got, want)
    say("  rel-L2 %.3e" % e)
    assert e <= TOL64
    s.clear()
