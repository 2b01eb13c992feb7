"""Resident fluid sweeps and the grid barriers of list rebuilds are never in
flight together on a card (each needs all its blocks placed): a solve takes one
launch per sweep while another context's call may enqueue rebuilds, an ensemble
steps its fluid boxes after its rebuilds, and the results are those of each
context alone, bit for bit."""
import threading
import time

import numpy
import pytest

import sphere_amd
from sphere_amd import _abi
from _cases import darcy_case, dense_case, settling_case

pytestmark = pytest.mark.gpu

KEYS = ("x", "vel", "force", "p_f")


def _fluid(ndem=1):
    s = darcy_case(n=900, seed=2, nxyz=(11, 7, 23), tolerance=1e-7, ndem=ndem)
    s.time_file_dt[0] = s.time_total[0] = 1.0
    return s


def _engine(s):
    e = sphere_amd.Engine(0)
    e.load(s.to_state())
    return e


def _afloat():
    s = settling_case(n=1000, seed=5, steps=100000)
    s.g[:] = 0.0
    s.angvel[:] = 1.0
    return s


def test_solve_beside_another_threads_rebuilds():
    ref, e = _engine(_fluid()), _engine(_fluid())
    grains, started = _engine(_afloat()), threading.Event()
    steps = 40000
    alone = _engine(_afloat())
    alone.step(steps)

    def run():
        started.set()
        grains.step(steps)

    t = threading.Thread(target=run)
    print("solves beside the steps of another thread", flush=True)
    t.start()
    started.wait()
    time.sleep(0.05)
    e.step(3)
    during = e.resident_stats()
    beside = t.is_alive()
    t.join()
    e.step(3)
    after = e.resident_stats()
    print("during", during.solves, during.yielded, "after", after.solves, after.yielded, flush=True)
    assert beside and (during.solves, during.repeated, during.yielded) == (0, 0, 3)
    assert (after.solves, after.repeated, after.yielded) == (3, 0, 3)
    ref.step(6)
    a, b = e.read().arrays, ref.read().arrays
    for k in KEYS:
        assert numpy.array_equal(a[k], b[k]), k
    a, b = grains.read().arrays, alone.read().arrays
    for k in KEYS[:3]:
        assert numpy.array_equal(a[k], b[k]), k


def test_ensemble_of_grains_and_single_fluid_boxes():
    """Boxes whose fluid the ensemble does not step together: two DEM steps per
    fluid step."""
    boxes = [dense_case(n=512, seed=0, model=3, periodic=1, nw=1, E=7e9), _fluid(ndem=2), settling_case(n=1500, seed=4),
             _fluid(ndem=2)]
    for s in boxes:
        s.time_file_dt[0] = s.time_total[0] = 1.0
    alone, together = [_engine(s) for s in boxes], [_engine(s) for s in boxes]
    ens = sphere_amd.Ensemble(together)
    for n in (5, 6):
        print("ensemble with single fluid boxes", n, flush=True)
        ens.step(n)
        for k, (e, r) in enumerate(zip(together, alone)):
            r.step(n)
            a, b = e.read().arrays, r.read().arrays
            for key in KEYS[:3] + (KEYS[3:] if k in (1, 3) else ()):
                assert numpy.array_equal(a[key], b[key]), (k, key)
    info = ens.info()
    assert info["multi_boxes"] == 2 and info["fluid_boxes"] == 0
    for k in (1, 3):
        rs = together[k].resident_stats()
        assert (rs.solves, rs.repeated, rs.yielded) == (6, 0, 0), k
    ens.close()
