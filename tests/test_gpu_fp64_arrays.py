"""FP64 arrays on mixed-precision solvers: the cell lists of the fixed-point
spreading are built with the positions (a product at fixed positions launches
no list kernels), and they follow the positions in every order of eager and
captured calls.  Integer sums do not depend on their order, so each result
equals that of a fresh solver at the same positions bit for bit; the spread
grid agrees with the FP64 oracle to the mixed-precision bound."""
import ctypes

import numpy as np
import pytest

from test_gpu_parity import rel_l2, say

pytestmark = pytest.mark.gpu

ETA = 1 / (6 * np.pi)
N, NX, NZ, LZ = 300, 32, 33, 12.0
L = 0.5 * NX
KINDS = ["forces", "torques", "regular"]


def _solver(kind):
    from doublyperiodicstokes_amd import DPStokes, StokesParameters
    par = StokesParameters(viscosity=ETA, Lx=L, Ly=L, zmin=0.0, zmax=LZ, w=6, w_d=0 if kind == "forces" else 5,
                           beta=1.785 * 6, beta_d=1.785 * 5, nx=NX, ny=NX, nz=NZ, mode="slit", precision="mixed",
                           useRegKernel=kind == "regular")
    s = DPStokes()
    s.initialize(par, N)
    return s


def _inputs(kind, seed=3):
    import torch
    rng = np.random.RandomState(seed)
    pos = [torch.tensor(np.stack([rng.uniform(0, L, N), rng.uniform(0, L, N), rng.uniform(0.3, LZ - 0.3, N)], 1).ravel(),
                        device="cuda") for _ in range(4)]
    F = torch.tensor(rng.normal(size=3 * N), device="cuda")
    T = None if kind == "forces" else torch.tensor(rng.normal(size=3 * N), device="cuda")
    return pos, F, T


def _fresh(kind, pos, F, T):
    s = _solver(kind)
    s.setPositions(pos)
    out = [None if a is None else a.cpu().numpy() for a in s.mdot_device(F, T)]
    s.clear()
    return out


def _same(got, want):
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert np.array_equal(a.cpu().numpy(), b)


def _kernel_nodes(graph):
    hip = ctypes.CDLL("libamdhip64.so")
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("kind", KINDS)
def test_products_build_no_lists(kind):
    """Launches of a captured product: with FP64 arrays those of FP32 arrays
    and, per spreading pass, the maxima that set the fixed-point scale."""
    import torch
    say("launches of a product with FP64 arrays, %s" % kind)
    pos, F, T = _inputs(kind)
    count = {}
    for dt in (torch.float32, torch.float64):
        s = _solver(kind)
        s.setPositions(pos[0])
        f, t = F.to(dt), None if T is None else T.to(dt)
        s.mdot_device(f, t)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(g):
            s.mdot_device(f, t)
        count[dt] = _kernel_nodes(g)
        s.clear()
    say("  FP32 arrays %d, FP64 arrays %d" % (count[torch.float32], count[torch.float64]))
    assert count[torch.float64] <= count[torch.float32] + (2 if kind == "regular" else 1)


@pytest.mark.parametrize("kind", KINDS)
def test_lists_follow_positions(kind):
    import torch
    say("FP64 arrays over changing positions, %s" % kind)
    pos, F, T = _inputs(kind)
    want = [_fresh(kind, p, F, T) for p in pos]
    wantF = [_fresh(kind, p, F, None) for p in pos]
    s = _solver(kind)
    for i in (0, 1):
        s.setPositions(pos[i])
        _same(s.mdot_device(F, T), want[i])
        _same(s.mdot_device(F, None), wantF[i])      # another pass at the same positions
        _same(s.mdot_device(F, T), want[i])
    work = pos[2].clone()
    s.update_positions_device(work, None, 0.0)
    _same(s.mdot_device(F, T), want[2])
    s.setPositions(pos[3].float())                   # positions in FP32 as well
    f32 = _fresh(kind, pos[3].float(), F, T)
    _same(s.mdot_device(F, T), f32)
    # a captured step (update, product) replayed on changing positions, with
    # eager products between the replays
    buf = pos[0].clone()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        s.update_positions_device(buf, None, 0.0, check=False)
        out = s.mdot_device(F, T)
    for i in (1, 2, 0, 3):
        buf.copy_(pos[i])
        g.replay()
        torch.cuda.synchronize()
        _same(out, want[i])
        _same(s.mdot_device(F, None), wantF[i])
        _same(s.mdot_device(F, T), want[i])
    # an eager set, then a replay of a captured product alone
    gp = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gp):
        outp = s.mdot_device(F, T)
    for i in (2, 1):
        s.setPositions(pos[i])
        gp.replay()
        torch.cuda.synchronize()
        _same(outp, want[i])
    s.clear()


@pytest.mark.parametrize("kind", KINDS)
def test_update_captured_before_the_first_product(kind):
    """A step captured by a solver that had seen FP32 arrays only builds no cell
    lists: products with FP64 arrays after its replays must not read old ones."""
    import torch
    say("update captured before the first product with FP64 arrays, %s" % kind)
    pos, F, T = _inputs(kind, 5)
    want = [_fresh(kind, p, F, T) for p in pos]
    s = _solver(kind)
    s.setPositions(pos[0])
    s.mdot_device(F.float(), None if T is None else T.float())
    buf = pos[0].clone()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        s.update_positions_device(buf, None, 0.0, check=False)
    _same(s.mdot_device(F, T), want[0])
    for i in (1, 2, 3):
        buf.copy_(pos[i])
        g.replay()
        _same(s.mdot_device(F, T), want[i])
        _same(s.mdot_device(F, T), want[i])
    s.setPositions(pos[1])
    _same(s.mdot_device(F, T), want[1])
    s.clear()


def test_chunks_change_under_captured_products():
    """A z chunk set after products were captured -- by the caller, and by two
    batches that share a solver -- leaves every replay right."""
    import torch
    from doublyperiodicstokes_amd import DPStokesBatch
    from doublyperiodicstokes_amd import _native as Nt
    say("z chunks changed under captured products")
    kind = "torques"
    pos, F, T = _inputs(kind, 7)
    want = _fresh(kind, pos[0], F, T)
    ok = lambda out: all(rel_l2(a.cpu().numpy(), b) <= 1e-6 for a, b in zip(out, want))
    set_chunk = lambda b, c: Nt.check(Nt.load().dps_batch_set_chunks(b._b, (ctypes.c_int * 1)(c), 1, None))
    s = _solver(kind)
    s.setPositions(pos[0])
    b1, b2 = DPStokesBatch([s]), DPStokesBatch([s])
    first = [[a[0].clone() for a in b.mdot_device([F], [T])] for b in (b1, b2)]
    assert all(ok(o) for o in first)
    for c in (8, 16, 12):
        set_chunk(b1, c)
        for b in (b2, b1):
            assert ok([a[0] for a in b.mdot_device([F], [T])])
        assert ok(s.mdot_device(F, T))
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        out = s.mdot_device(F, T)
    for c in (16, 8):
        set_chunk(b1, c)
        g.replay()
        torch.cuda.synchronize()
        assert ok(out) and ok(s.mdot_device(F, T)) and ok([a[0] for a in b2.mdot_device([F], [T])])
    b1.clear()
    b2.clear()
    s.clear()


@pytest.mark.parametrize("captured", ["first product", "update"])
def test_chunks_change_under_captured_builds(captured):
    """A z chunk set after a call that builds cell lists was captured: its
    replays must not leave lists of another chunk to the eager products."""
    import torch
    from doublyperiodicstokes_amd import DPStokesBatch
    from doublyperiodicstokes_amd import _native as Nt
    say("z chunks changed after capturing the %s" % captured)
    kind = "torques"
    pos, F, T = _inputs(kind, 9)
    want = [_fresh(kind, p, F, T) for p in pos[:2]]
    ok = lambda out, i: all(rel_l2(a.cpu().numpy(), b) <= 1e-6 for a, b in zip(out, want[i]))
    s = _solver(kind)
    s.setPositions(pos[0])
    if captured == "update":
        s.mdot_device(F, T)
    else:
        s.mdot_device(F.float(), T.float())
    buf = pos[0].clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        if captured == "update":
            s.update_positions_device(buf, None, 0.0, check=False)
        else:
            out = s.mdot_device(F, T)
    b = DPStokesBatch([s])
    for c in (8, 16, 12, 8):
        assert ok(s.mdot_device(F, T), 0)
        Nt.check(Nt.load().dps_batch_set_chunks(b._b, (ctypes.c_int * 1)(c), 1, None))
        for i in (1, 0):
            if captured == "update":
                buf.copy_(pos[i])
            else:
                s.setPositions(pos[i])
            g.replay()
            torch.cuda.synchronize()
            assert captured == "update" or ok(out, i)
            assert ok(s.mdot_device(F, T), i)
    b.clear()
    s.clear()


# name, mode, nx, ny, nz, particles, w, w_d, fraction of the box, size of the largest force
UNEVEN = [
    ("crowded_tile", "bottom", 64, 32, 33, 1500, 6, 6, 0.04, 1.0),
    ("crowded_two_kernels", "slit", 64, 32, 33, 1500, 6, 5, 0.06, 1.0),
    ("crowded_regular", "slit", 64, 32, 33, 1500, 6, 6, 0.05, 1.0),
    ("crowded_periodic", "periodic", 64, 32, 24, 2500, 5, 5, 0.1, 1.0),
    ("one_large_force", "slit", 64, 64, 33, 8000, 6, 6, 1.0, 100.0),
    ("one_large_force_in_a_tile", "bottom", 64, 32, 33, 8000, 6, 0, 0.05, 100.0),
    ("one_huge_force", "nowall", 48, 40, 30, 900, 5, 4, 1.0, 1e6),
]


@pytest.mark.parametrize("case", UNEVEN, ids=[c[0] for c in UNEVEN])
def test_crowded_and_uneven_grids(case):
    """Cells whose bound on the sums is far above them: the spread grid of FP64
    arrays holds the mixed-precision bound, rel-L2 <= 1e-5, and repeats bit for
    bit."""
    import torch
    from doublyperiodicstokes_amd import DPStokes, StokesParameters
    from oracle.dp_oracle import OracleDPStokes
    from oracle.tp_oracle import OracleTPStokes
    name, mode, nx, ny, nz, n, w, wd, box, top = case
    say("FP64 arrays, %s" % name)
    regular = name == "crowded_regular"
    h = 0.5
    Lx, Ly, Lz = h * nx, h * ny, (h * nz if mode == "periodic" else 0.35 * nz)
    rng = np.random.RandomState(n + nx)
    edge = 0.52 * max(w, wd) * h
    lo, hi = (edge if mode == "nowall" else 0.1), Lz - (edge if mode in ("nowall", "bottom") else 0.1)
    pos = np.stack([rng.uniform(0, box * Lx, n), rng.uniform(0, box * Ly, n), rng.uniform(lo, hi, n)], 1).ravel()
    F = rng.normal(size=3 * n)
    F[3 * (n // 2):3 * (n // 2) + 3] *= top
    T = rng.normal(size=3 * n) if wd else None
    has = wd > 0 and not regular
    kw = dict(has_torque=has, w_d=wd if has else None, betaw_d=1.785 * wd if has else None)
    if mode == "periodic":
        ref = OracleTPStokes(Lx, Ly, 0.0, Lz, nx, ny, nz, ETA, w, 1.785 * w, **kw)
    else:
        ref = OracleDPStokes(mode, Lx, Ly, 0.0, Lz, nx, ny, nz, ETA, w, 1.785 * w, **kw)
    ref.set_positions(pos)
    par = StokesParameters(viscosity=ETA, Lx=Lx, Ly=Ly, zmin=0.0, zmax=Lz, w=w, w_d=wd, beta=1.785 * w,
                           beta_d=1.785 * wd if wd else -1.0, nx=nx, ny=ny, nz=nz, mode=mode, precision="mixed",
                           useRegKernel=regular)
    s = DPStokes()
    s.initialize(par, n)
    s.setPositions(pos)
    for t in ([None, T] if has else [None]):
        got = s.stage_spread(torch.from_numpy(F), None if t is None else torch.from_numpy(t)).cpu().numpy()
        e = rel_l2(got, ref.spread_forces(F, t))
        say("  %s rel-L2 %.3e" % ("forces" if t is None else "forces and torques", e))
        assert e <= 1e-5
        s.setPositions(pos)
        assert np.array_equal(s.stage_spread(torch.from_numpy(F), None if t is None else torch.from_numpy(t)).cpu().numpy(), got)
    s.clear()
