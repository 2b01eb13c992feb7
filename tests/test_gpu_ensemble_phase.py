"""The first call of an ensemble hashes its boxes and steps once before the
pairs of steps; the pairs must still meet the rebuild and wrap flags of their
own steps: grains that cross the periodic faces and lists that are rebuilt
every few steps, in one call, against the oracle."""
import numpy
import pytest

import sphere_amd
from _cases import dense_case
from _oracle import Oracle
from _parity import compare_contacts, compare_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("steps", [2, 3, 30, 41])
def test_first_call_against_oracle(steps, graph):
    s = dense_case(n=512, seed=8, periodic=1, vmag=2.0)
    e = sphere_amd.Engine(0, skin=0.01)
    e.load(s.to_state())
    ens = sphere_amd.Ensemble([e])
    ens.set_graph(graph)
    print("ensemble, first call of", steps, "steps, graph", graph, flush=True)
    ora = Oracle(s.to_state(), nc=e.nc)
    ens.step(steps)
    ora.step(steps)
    compare_contacts(e, ora, steps)
    compare_state(e.read(), ora.read(), 512, steps, label="first call")
    assert steps < 30 or e.neighbor_stats().rebuilds >= 3
    del ens
    e.close()
