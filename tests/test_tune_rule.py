"""What dps_batch_tune times and what a stored chunk names (dps_tune.h,
compiled for the host): the launch in use is timed first and kept unless
another is clearly faster, every candidate differs in its launch, and the
chunk reported for a launch names that launch again."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def tune(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tune") / "libtune.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                           "-I", os.path.join(ROOT, "doublyperiodicstokes_amd", "csrc"),
                           "-o", out, os.path.join(ROOT, "tests", "native", "tune_check.cpp")])
    return ctypes.CDLL(out)


def own_chunk(tune, tsz, rs, nz):
    """The solver's chunk: 16 rows or all, halved until it fits."""
    zc = min(16, nz)
    while zc > 1 and not tune.tune_fits(tsz, rs, zc):
        zc //= 2
    return zc


@pytest.mark.parametrize("tsz,rs,nz", [(4, 60, 12), (4, 60, 48), (4, 110, 96), (4, 145, 96), (4, 200, 64),
                                       (4, 480, 128), (8, 60, 12), (8, 60, 48), (8, 110, 96), (8, 145, 96), (8, 200, 64)])
def test_tile_candidates(tune, tsz, rs, nz):
    max_tiles = 3 if tsz == 4 else 2
    own = own_chunk(tune, tsz, rs, nz)
    assert tune.tune_fits(tsz, rs, own)
    buf = (ctypes.c_int * 16)()
    for own_tiles in range(1, max_tiles + 1):
        n = tune.tune_tile_candidates(own_tiles, own, own_tiles, max_tiles, tsz, rs, nz, buf)
        cand = [(buf[2 * i], buf[2 * i + 1]) for i in range(n)]
        assert cand[0] == (own, own_tiles)
        assert len({t for _, t in cand}) == n
        for now in [t for _, t in cand]:   # after an earlier choice: that one first, the same others
            m = tune.tune_tile_candidates(now, own, own_tiles, max_tiles, tsz, rs, nz, buf)
            again = [(buf[2 * i], buf[2 * i + 1]) for i in range(m)]
            assert again[0][1] == now and sorted(again) == sorted(cand)
        for c, t in cand:
            assert tune.tune_tiles(c, own, own_tiles, max_tiles) == t and tune.tune_fits(tsz, rs, c) and c <= nz


def test_two_tiles_are_a_choice_in_fp64(tune):
    """256 x 256 x 96 in FP64: only chunks up to 12 rows fit, and two tiles per
    wavefront are the solver's own launch."""
    buf = (ctypes.c_int * 16)()
    n = tune.tune_tile_candidates(2, 8, 2, 2, 8, 110, 96, buf)
    assert [(buf[2 * i], buf[2 * i + 1]) for i in range(n)] == [(8, 2), (12, 1)]
    assert tune.tune_tiles(8, 8, 2, 2) == 2


@pytest.mark.parametrize("now,rs,nz", [(16, 110, 96), (8, 145, 96), (13, 60, 13), (32, 60, 40)])
def test_chunk_candidates(tune, now, rs, nz):
    buf = (ctypes.c_int * 16)()
    c = list(buf[:tune.tune_chunk_candidates(now, 4, rs, nz, buf)])
    assert c[0] == now and len(set(c)) == len(c) and all(x <= nz for x in c[1:])
    assert {x for x in (8, 12, 16) if x <= nz} <= set(c)


def test_the_launch_in_use_stays_unless_beaten(tune):
    pick = lambda *ms: tune.tune_fastest((ctypes.c_float * len(ms))(*ms), len(ms))  # noqa: E731
    assert pick(1.0) == 0
    assert pick(1.0, 0.99, 1.2) == 0
    assert pick(1.0, 0.9, 0.95) == 1
    assert pick(1.0, 0.97, 0.9) == 2
