"""Walls of a state without grains: a step integrates the walls only where
there are grains, so a wall of any mode keeps its position and velocity, also
one without mass (totalMass() of no grains), and the fluid under it sees the
same wall at each output event.  Against the oracle, bit for bit."""
import numpy
import pytest

import sphere_amd
from _cases import darcy_empty
from _oracle import Oracle

pytestmark = pytest.mark.gpu


def _box(wmode, mass, outputs):
    s = darcy_empty(p_top=10.0)
    s.nw[0] = 1
    s.wmode = numpy.array([wmode], dtype=numpy.int32)
    s.w_n = numpy.array([[0.0, 0.0, -1.0]])
    s.w_x = numpy.array([0.31])
    s.w_m = numpy.array([mass])
    s.w_vel = numpy.array([0.0])
    s.w_force = numpy.array([0.0])
    s.w_sigma0 = numpy.array([1.0e4])
    s.time_file_dt[0] = s.time_dt[0] * (2.5 if outputs else 1.0e6)
    return s


@pytest.mark.parametrize("wmode,mass,outputs", [(1, 1.0, False), (1, 0.0, False), (1, 0.0, True), (2, 1.0, True),
                                                (3, 1.0, True)])
def test_walls_stay(wmode, mass, outputs):
    s = _box(wmode, mass, outputs)
    print("walls without grains, mode", wmode, "mass", mass, "outputs", outputs, flush=True)
    e = sphere_amd.Engine(0)
    e.load(s.to_state())
    ora = Oracle(s.to_state())
    for _ in range(4):
        e.step(3)
        ora.step(3)
    g, o = e.read(), ora.read()
    assert g.state.w_nx[3] == o.state.w_nx[3] == 0.31
    for k in range(4):
        assert g.state.w_mvfd[k] == o.state.w_mvfd[k], k
    assert g.state.time_current == o.state.time_current
    cells = int(numpy.prod(s.num))
    for name in ("p_f", "phi", "dphi"):
        assert numpy.array_equal(g.get(name, cells, 1), o.get(name, cells, 1)), name
    e.close()
