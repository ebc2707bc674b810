"""Spread grids against the oracles where a wavefront holds two or three
16-level z tiles (large grids; 1 in the small ones of test_gpu_spread): last
groups with fewer tiles, last tiles with fewer rows, columns past the last
multiple of 4 and of the 32 x 4-column tiles, forces alone and with torques,
and levels or columns that wrap.  Bounds as there, rel-L2 of the grid <= 1e-11
in FP64 and <= 1e-5 in mixed precision; the expected tiles per wavefront are
those of spread_tiles."""
import numpy as np
import pytest

from oracle.dp_oracle import OracleDPStokes
from oracle.tp_oracle import OracleTPStokes
from test_gpu_parity import say
from test_gpu_spread import check

pytestmark = pytest.mark.gpu

ETA = 1 / (6 * np.pi)
# mode, nx, ny, nz, w, w_d, z tiles per wavefront in FP32 and FP64
CASES = [
    ("bottom", 258, 254, 50, 6, 6, 2, 2),
    ("slit", 258, 254, 70, 6, 5, 3, 2),
    ("nowall", 254, 258, 45, 5, 5, 3, 2),
    ("slit", 230, 234, 100, 6, 0, 3, 2),
    ("periodic", 142, 130, 83, 6, 6, 2, 2),
    ("periodic", 162, 158, 83, 5, 6, 3, 2),
    ("slit", 4, 12808, 20, 2, 0, 2, 2),
]


def tiles(nx, ny, nz, fp32):
    waves, zt = -(-nx // 4) * -(-ny // 4), -(-nz // 16)
    nt = 3 if fp32 else 2
    while nt > 1 and (waves * -(-zt // nt) < 3200 or -(-zt // (nt - 1)) == -(-zt // nt)):
        nt -= 1
    return nt


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("case", CASES, ids=["%s_%dx%dx%d" % c[:4] for c in CASES])
def test_spread_grid_matches_oracle(case, precision):
    import torch
    from doublyperiodicstokes_amd import DPStokes, StokesParameters
    mode, nx, ny, nz, w, wd, n32, n64 = case
    assert (tiles(nx, ny, nz, True), tiles(nx, ny, nz, False)) == (n32, n64)
    say("spread %s %dx%dx%d %s" % (case[:4] + (precision,)))
    h, N = 0.5, 400
    Lx, Ly, Lz = h * nx, h * ny, (h * nz if mode == "periodic" else 0.35 * nz)
    rng = np.random.RandomState(nx + nz)
    reach = 0.52 * max(w, wd) * h
    lo, hi = (reach if mode == "nowall" else 0.0), Lz - (reach if mode in ("nowall", "bottom") else 0.0)
    pos = np.stack([rng.uniform(0, Lx, N), rng.uniform(0, Ly, N), rng.uniform(lo, hi, N)], 1)
    # a few at the ends of the cell, some together
    pos[:40, :2] = np.array([Lx, Ly]) - rng.uniform(1e-9, 1.2, (40, 2)) * (rng.uniform(size=(40, 2)) < 0.7)
    pos[40:80, :2] = rng.uniform(1e-9, 1.2, (40, 2))
    pos[:, :2] %= [Lx, Ly]
    pos = pos.ravel()
    F = rng.normal(size=3 * N)
    T = rng.normal(size=3 * N) if wd else None
    kw = dict(has_torque=wd > 0, w_d=wd or None, betaw_d=1.785 * wd if wd else None)
    if mode == "periodic":
        ref = OracleTPStokes(Lx, Ly, 0.0, Lz, nx, ny, nz, ETA, w, 1.785 * w, **kw)
    else:
        ref = OracleDPStokes(mode, Lx, Ly, 0.0, Lz, nx, ny, nz, ETA, w, 1.785 * w, **kw)
    ref.set_positions(pos)
    par = StokesParameters(viscosity=ETA, Lx=Lx, Ly=Ly, zmin=0.0, zmax=Lz, w=w, w_d=wd, nx=nx, ny=ny, nz=nz,
                           beta=1.785 * w, beta_d=1.785 * wd if wd else -1.0, mode=mode, precision=precision)
    s = DPStokes()
    s.initialize(par, N)
    s.setPositions(pos)
    dt = torch.float64 if precision == "double" else torch.float32
    check(s, ref, torch.as_tensor(F, dtype=dt), None if T is None else torch.as_tensor(T, dtype=dt), F, T, pos,
          1e-11 if precision == "double" else 1e-5)
    s.clear()
