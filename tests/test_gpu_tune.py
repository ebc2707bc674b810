"""Tuning leaves a batch no slower than it found it: the spreading stage of a
solver whose default launch is the faster one (two z tiles in FP64), and of a
mixed-precision solver with FP64 arrays (rows of the fixed-point cells), with
the solver's own chunk and after dps_batch_tune (the shortest of 30 each, 10 %
for the timing, the best of three comparisons); and the chunks it reports are
accepted and give the same products."""
import ctypes

import numpy as np
import pytest

from test_gpu_parity import rel_l2, say

pytestmark = pytest.mark.gpu

ETA = 1 / (6 * np.pi)


@pytest.mark.parametrize("precision,arrays", [("double", "float64"), ("mixed", "float64"), ("mixed", "float32")])
def test_tuning_does_not_slow_the_spreading(precision, arrays, tmp_path):
    import torch
    from doublyperiodicstokes_amd import DPStokes, DPStokesBatch, StokesParameters
    from doublyperiodicstokes_amd import _native as Nt
    say("tuning, %s, %s arrays" % (precision, arrays))
    nx, nz, N, Lz = 256, 96, 16384, 32.0
    par = StokesParameters(viscosity=ETA, Lx=128.0, Ly=128.0, zmin=0.0, zmax=Lz, w=6, w_d=6, beta=1.785 * 6,
                           beta_d=1.785 * 6, nx=nx, ny=nx, nz=nz, mode="slit", precision=precision)
    s = DPStokes()
    s.initialize(par, N)
    rng = np.random.RandomState(2)
    dt = getattr(torch, arrays)
    dev = lambda a: torch.tensor(a, dtype=dt, device="cuda")
    s.setPositions(dev(np.stack([rng.uniform(0, 128, N), rng.uniform(0, 128, N), rng.uniform(0.5, Lz - 0.5, N)], 1).ravel()))
    F, T = dev(rng.normal(size=3 * N)), dev(rng.normal(size=3 * N))

    def spread_us():
        s.set_profiling(True)
        best = 1e9
        for _ in range(30):
            s.mdot_device(F, T)
            torch.cuda.synchronize()
            best = min(best, s.timings()["spread"])
        s.set_profiling(False)
        return best

    before, ref = spread_us(), s.mdot_device(F, T)[0].double().cpu().numpy()
    b = DPStokesBatch([s])
    path = str(tmp_path / "tune.json")
    chunks = b.tune([F], [T], cache=path)
    after = spread_us()
    own = (ctypes.c_int * 1)(8 if precision == "double" else 16)
    for _ in range(2):
        if after <= 1.10 * before:
            break
        Nt.check(Nt.load().dps_batch_set_chunks(b._b, own, 1, None))
        before = spread_us()
        assert b.tune([F], [T], cache=path) == chunks
        after = spread_us()
    say("  spread %.1f us, tuned %s %.1f us" % (before, chunks, after))
    assert after <= 1.10 * before
    assert b.tune([F], [T], cache=path) == chunks      # applied from the file
    assert rel_l2(s.mdot_device(F, T)[0].double().cpu().numpy(), ref) <= (1e-12 if precision == "double" else 1e-6)
    b.clear()
    s.clear()
