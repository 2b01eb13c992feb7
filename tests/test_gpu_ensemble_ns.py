"""A box with an attached Navier-Stokes fluid in an ensemble: it steps by
itself, with its fluid, beside the boxes stepped together, and grains and fluid
are those of the box alone, bit for bit; attached and detached between calls."""
import numpy
import pytest

import sphere_amd
from sphere_amd import _abi
from _cases import dense_case

pytestmark = pytest.mark.gpu


def _pair(s):
    nx, ny, nz = (int(v) for v in s.num)
    P = _abi.ns_params(nx, ny, nz, s.L, float(s.time_dt[0]), mu=1.0e-3, rho_f=1000.0, g=s.g, bc_bot=1, bc_top=0,
                       tolerance=1e-6, maxiter=3000)
    v = 0.01 * numpy.random.default_rng(6).standard_normal((nx, ny, nz, 3))
    e = sphere_amd.Engine(0)
    e.load(s.to_state())
    return e, sphere_amd.NavierStokes(P, v, numpy.zeros((nx, ny, nz)))


def test_attached_fluid_in_an_ensemble():
    wet = dense_case(n=343, seed=4, periodic=1, spacing_factor=1.02)
    dry = dense_case(n=512, seed=5, model=3, periodic=1, nw=1, E=7e9)
    (a, na), (b, nb) = _pair(wet), _pair(wet)
    others = [sphere_amd.Engine(0) for _ in range(2)]
    for e in others:
        e.load(dry.to_state())
    ens = sphere_amd.Ensemble([a, others[0]])
    for steps, fluid in ((3, True), (4, False), (2, True)):
        a.attach_fluid(na if fluid else None)
        b.attach_fluid(nb if fluid else None)
        print("ensemble,", steps, "steps, attached fluid", fluid, flush=True)
        ens.step(steps)
        b.step(steps)
        others[1].step(steps)
        assert na.stats().steps == nb.stats().steps
        for x, y in zip(na.read(), nb.read()):
            assert numpy.array_equal(x, y)
        for x, y in ((a, b), (others[0], others[1])):
            p, q = x.read().arrays, y.read().arrays
            for k in ("x", "vel", "force", "angvel"):
                assert numpy.array_equal(p[k], q[k]), (steps, k)
    assert na.stats().steps == 5
    ens.close()
    for e in (a, b):
        e.attach_fluid(None)
