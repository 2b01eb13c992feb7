"""Jacobi iterations in resident launches (resident.h) against the CPU
oracle: grids at the edges of the tile rules (the smallest, axes shorter than
a tile, uneven tiles, one and two cells per thread, one grid past the largest
that fits), periodic and closed z, solves that end at a test and at maxiter;
and the path a wait that runs out takes, forced by a bound of one poll, in the
first launch of a solve and in later ones.  Both paths give the same bits, so
every test reads from the solve statistics which one ran."""
import numpy
import pytest

import sphere_amd
from sphere_amd import _abi
from _cases import darcy_case
from _ns_oracle import NsOracle
from _parity import run_pair

pytestmark = pytest.mark.gpu

# cells that fit: 256 compute units, two cells on each of 960 threads
CELLS = 256 * 2 * 960


@pytest.mark.parametrize("shape,bb,bt,maxiter", [
    ((3, 3, 3), 1, 0, 500), ((3, 4, 61), 2, 2, 300), ((37, 3, 5), 1, 1, 47), ((17, 13, 9), 0, 0, 400),
    ((31, 33, 29), 1, 0, 61), ((33, 31, 30), 2, 2, 40), ((48, 50, 101), 1, 0, 31), ((64, 60, 110), 0, 1, 21),
    ((80, 64, 100), 1, 0, 12),
])
def test_ns_tiles(shape, bb, bt, maxiter):
    rng = numpy.random.default_rng(sum(shape))
    P = _abi.ns_params(*shape, [0.02 * n for n in shape], 2.0e-4, mu=1.0e-3, rho_f=1000.0,
                       g=(0.0, 0.0, -9.81), bc_bot=bb, bc_top=bt, tolerance=1e-6, maxiter=maxiter)
    v = 0.02 * rng.standard_normal(shape + (3,))
    p = 500.0 + 100.0 * rng.standard_normal(shape)
    print("ns tiles", shape, bb, bt, flush=True)
    gpu, ora = sphere_amd.NavierStokes(P, v, p), NsOracle(P, v, p)
    for step in range(2):
        gpu.step(1)
        ora.step(1)
        sg, so = gpu.stats(), ora.stats()
        assert (sg.iterations, sg.nonconverged, sg.last_nijac, sg.last_max_norm) == \
            (so.iterations, so.nonconverged, so.last_nijac, so.last_max_norm), step
        assert numpy.array_equal(gpu.field(3), ora.field(NsOracle.EPS)), step
    for a, b in zip(gpu.read(), ora.read()):
        assert numpy.array_equal(a, b)
    rs = gpu.resident_stats()
    assert (rs.solves, rs.repeated) == (2 if numpy.prod(shape) <= CELLS else 0, 0)
    gpu.close()


@pytest.mark.parametrize("nxyz,n,periodic,bc_bot,bc_top,tolerance", [
    ((3, 3, 7), 50, 1, 1, 0, 1e-8), ((5, 9, 8), 200, 1, 0, 0, 1e-6), ((11, 7, 23), 900, 0, 1, 0, 1e-7),
    ((18, 17, 21), 3000, 1, 1, 1, 1e-5),
])
def test_darcy_tiles(nxyz, n, periodic, bc_bot, bc_top, tolerance):
    s = darcy_case(n=n, seed=sum(nxyz), nxyz=nxyz, periodic=periodic, bc_bot=bc_bot, bc_top=bc_top,
                   tolerance=tolerance)
    e = sphere_amd.Engine(0)
    print("darcy tiles", nxyz, flush=True)
    ora, _ = run_pair(e, s, 2, 2, fluid=True, label="darcy tiles")
    assert e.darcy_stats().sweeps == ora.darcy_stats().sweeps
    rs = e.resident_stats()
    assert (rs.solves, rs.repeated) == (4, 0)
    e.close()


def test_wait_bound_falls_back():
    """A solve whose waits run out is repeated with one launch per sweep, bit
    for bit the solve it replaces, and so are the solves after it."""
    s = darcy_case(n=900, seed=2, nxyz=(11, 7, 23), tolerance=1e-7)
    got = []
    for spin in (0, 1):
        e = sphere_amd.Engine(0)
        e.set_barrier_spin_limit(spin)
        e.load(s.to_state())
        print("darcy, wait bound", spin, flush=True)
        e.step(3)
        got.append((e.read().arrays, e.darcy_stats().sweeps))
        rs = e.resident_stats()
        assert (rs.solves, rs.repeated) == ((3, 0) if spin == 0 else (0, 1))
        e.close()
    assert got[0][1] == got[1][1]
    for k in ("p_f", "x", "vel", "force"):
        assert numpy.array_equal(got[0][0][k], got[1][0][k]), k


def test_resident_again_after_a_pause():
    """After a wait has run out 16 solves, then 32, take one launch per sweep,
    and the next one is resident again."""
    s = darcy_case(n=200, seed=3, nxyz=(5, 9, 8), tolerance=1e-7)
    ref, e = sphere_amd.Engine(0), sphere_amd.Engine(0)
    ref.load(s.to_state())
    e.load(s.to_state())
    for polls, steps, want in ((1, 17, (0, 1)), (1, 1, (0, 2)), (0, 32, (0, 2)), (0, 2, (2, 2))):
        e.set_resident_wait_limit(polls)
        print("darcy, wait bound", polls, steps, "steps", flush=True)
        e.step(steps)
        rs = e.resident_stats()
        assert (rs.solves, rs.repeated) == want
    ref.step(52)
    assert ref.resident_stats().solves == 52 and ref.darcy_stats().sweeps == e.darcy_stats().sweeps
    a, b = e.read().arrays, ref.read().arrays
    for k in ("p_f", "x", "vel", "force"):
        assert numpy.array_equal(a[k], b[k]), k
    e.close()
    ref.close()


@pytest.mark.parametrize("learned,later", [(True, 2), (True, 12), (True, 22), (False, 20000)])
def test_wait_bound_in_a_later_launch(learned, later):
    """A wait that runs out after earlier launches of the solve have written
    both iterate buffers, with the learned correction between them or past the
    sweeps of one launch: the repeated solve starts where the first did."""
    from sphere_amd import learn
    s = darcy_case(n=700, seed=4, nxyz=(8, 8, 16), tolerance=1e-7 if learned else -1.0,
                   maxiter=20000 if learned else 20025)
    s.p_f[:] = 10.0 * numpy.random.default_rng(3).standard_normal(s.p_f.shape)
    got = []
    for polls, first in ((0, 0), (1, 0), (1, later)):
        e = sphere_amd.Engine(0)
        e.load(s.to_state())
        e.set_resident_wait_limit(polls, first)
        if learned:
            e.set_darcy_net(learn.init_params(1), max_corrections=5)
        print("darcy, wait bound", polls, "from sweep", first, "learned", learned, flush=True)
        e.step(1)
        st, rs = e.darcy_stats(), e.resident_stats()
        assert (rs.solves, rs.repeated) == ((1, 0) if polls == 0 else (0, 1))
        assert st.corrections == (5 if learned else 0) and st.sweeps > later
        got.append((e.read().arrays, st.sweeps, st.corrections, st.last_max_residual))
        e.close()
    for g in got[1:]:
        assert g[1:] == got[0][1:]
        for k in ("p_f", "x", "vel", "force"):
            assert numpy.array_equal(got[0][0][k], g[0][k]), k


@pytest.mark.parametrize("later", [0, 20000])
def test_ns_wait_bound_falls_back(later):
    """In the first launch, and in the one past the 20,000 iterations of a
    launch, on a column too tall to have converged by then."""
    from _cases import dense_case
    s = dense_case(n=343, seed=4, periodic=1, vmag=0.0, wmag=0.0, spacing_factor=1.1)
    if later:
        s.L[2] *= 400.0 / s.num[2]
        s.num[2] = 400
    nx, ny, nz = (int(v) for v in s.num)
    P = _abi.ns_params(nx, ny, nz, s.L, float(s.time_dt[0]), mu=1.0e-3, rho_f=1000.0, g=s.g,
                       bc_bot=1, bc_top=0, tolerance=-1.0 if later else 1e-10, maxiter=20044)
    v = 0.002 * numpy.random.default_rng(6).standard_normal((nx, ny, nz, 3))
    got = []
    for polls, first in ((0, 0), (1, later)):
        e = sphere_amd.Engine(0)
        e.set_resident_wait_limit(polls, first)
        e.load(s.to_state())
        ns = sphere_amd.NavierStokes(P, v, numpy.zeros((nx, ny, nz)))
        e.attach_fluid(ns)
        print("ns, wait bound", polls, "from iteration", first, flush=True)
        e.step(3)
        rs = ns.resident_stats()
        assert (rs.solves, rs.repeated) == ((3, 0) if polls == 0 else (0, 1))
        st = ns.stats()
        assert st.iterations == 3 * 20044 and st.last_max_norm > 0.0 if later else st.iterations < 3 * 20044
        got.append((ns.read(), (st.iterations, st.last_max_norm), e.read().arrays["vel"]))
        e.attach_fluid(None)
        e.close()
    for g in got[1:]:
        assert g[1] == got[0][1]
        for a, b in zip(got[0][0], g[0]):
            assert numpy.array_equal(a, b)
        assert numpy.array_equal(got[0][2], g[2])
