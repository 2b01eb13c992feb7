"""Neighbour lists under a Darcy fluid: the cell sort runs every step, the
lists are rebuilt only where grains have moved, and the hash of the next step
lies beside the sorted keys.  Cells, sort, contact rows and state against the
oracle over steps in which grains wrap and lists are kept and rebuilt; and a
box stepped alone, in an ensemble (which hashes and rebuilds every step) and
alone again."""
import numpy
import pytest

import sphere_amd
from _cases import darcy_case
from _oracle import Oracle
from _parity import compare_contacts, compare_sort, compare_state, run_pair

pytestmark = pytest.mark.gpu


N = 294


def _moving(seed):
    """Grains apart from each other on a lattice, at up to 4 m/s per axis
    (17 um a step), the outer ones next to the periodic faces."""
    rng = numpy.random.default_rng(seed)
    s = darcy_case(n=N, seed=seed, nxyz=(6, 7, 12), tolerance=1e-6, ndem=4)
    g = numpy.arange(N)
    s.x[:] = 0.0231 * (numpy.stack([g % 6, g // 6 % 7, g // 42 + 1], axis=1) + 0.02)
    s.x[:] += rng.uniform(0.0, 3e-4, s.x.shape)
    s.vel[:] = rng.uniform(-4.0, 4.0, s.vel.shape)
    return s


@pytest.mark.parametrize("skin,fused", [(0.02, True), (0.1, True), (0.1, False)])
def test_lists_kept_under_fluid(skin, fused):
    e = sphere_amd.Engine(0, skin=skin, fused_rebuild=fused)
    print("fluid lists, skin", skin, flush=True)
    s = _moving(5)
    run_pair(e, s, 8, 5, fluid=True, label="fluid lists")
    st = e.neighbor_stats()
    assert 1 <= st.rebuilds < 40
    x = e.read().get("x", N, 4)
    assert numpy.any(numpy.abs(x[:, :2] - s.x[:, :2]) > 0.05)  # some wrapped
    e.close()


def test_alone_and_in_an_ensemble():
    s = _moving(6)
    e = sphere_amd.Engine(0, skin=0.02)
    e.load(s.to_state())
    ora = Oracle(s.to_state(), nc=e.nc)
    ens = sphere_amd.Ensemble([e])
    print("fluid lists, alone and in an ensemble", flush=True)
    done = 0
    for step, n in ((e.step, 7), (ens.step, 3), (e.step, 6), (ens.step, 4), (e.step, 5)):
        step(n)
        ora.step(n)
        done += n
        compare_sort(e, ora)
        compare_contacts(e, ora, done)
        compare_state(e.read(), ora.read(), N, done, fluid=True, label="ensemble")
    del ens
    e.close()
