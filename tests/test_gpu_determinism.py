"""Bitwise reproducibility of the mixed-precision path.

The spreading sums run in particle order (each tile's list is sorted); the
FFTs, the spectral solve and the interpolation's wavefront reductions have
fixed orders.  So repeated calls on the same inputs give identical bits: the
spread grid, U and W, for forces only and with torques, with the
self-mobility's particle on a grid node and for a many-particle slit.
"""
import numpy as np
import pytest

from test_gpu_parity import CASES, gpu_for, make_case, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [CASES[2], CASES[6], CASES[5]], ids=[CASES[2][0], CASES[6][0], CASES[5][0]])
def test_mixed_precision_is_bitwise_reproducible(case):
    import torch
    say("case %s: repeated mixed-precision calls" % case[0])
    pos, F, T = make_case(case, seed=11)
    s = gpu_for(case, "mixed")
    s.setPositions(pos)
    dev = torch.device("cuda", 0)
    Fd = torch.tensor(F, dtype=torch.float32, device=dev)
    Td = torch.tensor(T, dtype=torch.float32, device=dev) if T is not None else None
    grids, outs = [], []
    for _ in range(4):
        grids.append(s.stage_spread(Fd, Td).cpu().numpy())
        U, W = s.mdot_device(Fd, Td)
        outs.append((U.cpu().numpy(), None if W is None else W.cpu().numpy()))
    for g in grids[1:]:
        assert np.array_equal(g, grids[0])
    for U, W in outs[1:]:
        assert np.array_equal(U, outs[0][0])
        if W is not None:
            assert np.array_equal(W, outs[0][1])
    say("  4 calls: spread grid, U%s identical" % (" and W" if T is not None else ""))
    s.clear()


def test_slit_workload_is_bitwise_reproducible():
    import torch
    import bench
    wl = bench.WORKLOADS["slit16k"]
    say("workload slit16k: repeated mixed-precision Mdot")
    pos, F, T = bench.make_inputs(wl)
    s = bench.gpu_solver(wl, "mixed")
    s.setPositions(pos)
    dev = torch.device("cuda", 0)
    Fd = torch.from_numpy(F.astype(np.float32)).to(dev)
    Td = torch.from_numpy(T.astype(np.float32)).to(dev)
    U0, W0 = [t.cpu().numpy() for t in s.mdot_device(Fd, Td)]
    for _ in range(3):
        U, W = [t.cpu().numpy() for t in s.mdot_device(Fd, Td)]
        assert np.array_equal(U, U0) and np.array_equal(W, W0)
    s.clear()
