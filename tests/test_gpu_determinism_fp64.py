"""Repeated products of an FP64 solver, over repeated builds of the same
positions, give the same bits: the spreading sums run in particle order, and
every later stage has a fixed order."""
import numpy as np
import pytest

from test_gpu_parity import CASES, gpu_for, make_case, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [CASES[2], CASES[6], CASES[5]], ids=[CASES[2][0], CASES[6][0], CASES[5][0]])
def test_fp64_is_bitwise_reproducible(case):
    import torch
    say("case %s: repeated FP64 calls" % case[0])
    pos, F, T = make_case(case, seed=11)
    s = gpu_for(case, "double")
    Fd = torch.tensor(F, dtype=torch.float64, device="cuda")
    Td = torch.tensor(T, dtype=torch.float64, device="cuda") if T is not None else None
    first = None
    for _ in range(3):
        s.setPositions(pos)
        for _ in range(2):
            out = [a.cpu().numpy() for a in s.mdot_device(Fd, Td) if a is not None] + [s.stage_spread(Fd, Td).cpu().numpy()]
            first = out if first is None else first
            assert all(np.array_equal(a, b) for a, b in zip(out, first))
    s.clear()
