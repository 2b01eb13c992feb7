"""The last boxes of an ensemble's Darcy solves go on in resident launches: states,
pressures, sweep and correction counts are those of each box alone, bit for bit,
whether the long solve ends at a test or at maxiter, in one launch or in
several, with the learned correction before it, with a wait that runs out in
its first or a later launch, or where a flux boundary rules them out."""
import numpy
import pytest

import sphere_amd
from _cases import darcy_case

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vel", "force", "p_f", "phi", "v_f")


def _box(k, long, maxiter=20000, flux=False, shape=(8, 8, 16)):
    s = darcy_case(n=300, seed=k, nxyz=shape, tolerance={0: 1e-5, 1: 1e-12, 2: -1.0}[long], maxiter=maxiter,
                   bc_top=4 if flux else 0)
    s.p_f[:] = 10.0 * numpy.random.default_rng(k).standard_normal(s.p_f.shape)
    if flux:
        s.bc_top_flux[0] = 1e-6
    s.time_file_dt[0] = s.time_total[0] = 1.0
    return s


# the long solves' kind (0 short, 1 to 1e-12, 2 to maxiter), boxes with the
# network, boxes with a flux boundary, wait bound and its first sweep, the
# solves per step in resident launches per box, and those repeated in all
CASES = {
    "one long": dict(long=[0, 1, 0, 0], want=[0, 1, 0, 0]),
    "two long": dict(long=[1, 0, 0, 1], want=[1, 0, 0, 1]),
    "two boxes": dict(long=[0, 1], want=[1, 1]),
    "learned": dict(long=[0, 0, 1, 0], learned=[0, 2], want=[0, 0, 1, 0]),
    "flux": dict(long=[0, 1, 0], flux=[1], want=[0, 0, 0]),
    "flux beside": dict(long=[0, 1, 0], flux=[0], want=[0, 1, 0]),
    "maxiter": dict(long=[0, 0, 2], maxiter=1235, want=[0, 0, 1]),
    "chunks": dict(long=[0, 2, 0], maxiter=20531, steps=(2,), want=[0, 1, 0]),
    "wait": dict(long=[0, 1, 0, 1], wait=(1, 0), want=[0, 0, 0, 0], repeated=2),
    "later wait": dict(long=[0, 2, 0], maxiter=20531, steps=(2,), wait=(1, 20000), want=[0, 0, 0], repeated=1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_last_boxes(name):
    from sphere_amd import learn
    c = CASES[name]
    boxes = [_box(k, kind, c.get("maxiter", 20000), k in c.get("flux", ()), (8, 8, 16) if k != 1 else (7, 6, 17))
             for k, kind in enumerate(c["long"])]
    params = learn.init_params(3)

    def engines(wait):
        out = []
        for k, s in enumerate(boxes):
            e = sphere_amd.Engine(0, nc=64)
            if k in c.get("learned", ()):
                e.set_darcy_net(params, 4)
            e.load(s.to_state())
            e.set_resident_wait_limit(*wait)
            out.append(e)
        return out

    together, alone = engines(c.get("wait", (0, 0))), engines((0, 0))
    ens = sphere_amd.Ensemble(together)
    total = 0
    for steps in c.get("steps", (3, 2)):
        print("ensemble,", name, steps, "steps", flush=True)
        ens.step(steps)
        total += steps
        for k, (a, b) in enumerate(zip(together, alone)):
            b.step(steps)
            sa, sb = a.darcy_stats(), b.darcy_stats()
            assert (sa.sweeps, sa.corrections, sa.nonconverged, sa.last_nijac, sa.last_max_residual) == \
                (sb.sweeps, sb.corrections, sb.nonconverged, sb.last_nijac, sb.last_max_residual), k
            p, q = a.read().arrays, b.read().arrays
            for f in FIELDS:
                assert numpy.array_equal(p[f], q[f]), (k, f)
    assert ens.info()["fluid_boxes"] == len(boxes)
    rs = [e.resident_stats() for e in together]
    print([(r.solves, r.repeated, r.yielded) for r in rs], flush=True)
    # a short solve may be among the last two as well
    for r, kind, want in zip(rs, c["long"], c["want"]):
        assert r.solves == want * total if kind else r.solves <= (0 if "wait" in c else total)
    assert sum(r.repeated for r in rs) == c.get("repeated", 0) and sum(r.yielded for r in rs) == 0
    ens.close()
