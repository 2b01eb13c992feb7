"""State reads through the pinned staging memory that all contexts share: the
same arrays as straight to the destination (the path where no pinned memory can
be had), at sizes on both sides of the one-wait copy (4 MB) and of the piece
sizes, after loads of larger and smaller states, and from several threads at
once; the memory is given back with the last context and made anew."""
import threading

import numpy
import pytest

import sphere_amd

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vel", "angvel", "force", "torque", "angpos", "xyzsum", "es_dot", "es", "ev_dot", "ev", "p")


def _state(n, seed):
    """n grains apart from each other on a lattice, every particle array random."""
    rng = numpy.random.default_rng(seed)
    side = int(numpy.ceil(n ** (1.0 / 3.0)))
    s = sphere_amd.sim(np=n, sid="read", nw=0)
    s.radius[:] = 0.01
    g = numpy.arange(n)
    s.x[:] = 0.03 * numpy.stack([g % side, g // side % side, g // side ** 2], axis=1) + 0.03
    for a in (s.vel, s.angvel, s.force, s.torque, s.angpos, s.xyzsum, s.es_dot, s.es, s.ev_dot, s.ev, s.p):
        a[:] = rng.standard_normal(a.shape)
    s.defaultParams()
    s.defineWorldBoundaries(L=[0.03 * (side + 2)] * 3)
    s.initTemporal(total=1.0, file_dt=1.0, dt=1e-6)
    return s


def _same(got, s, n):
    ref = s.to_state()
    for k in FIELDS:
        assert numpy.array_equal(got.arrays[k], ref.arrays[k]), (n, k)


@pytest.mark.parametrize("sizes", [[1], [1000, 18000, 19000], [100000, 1000, 90001]])
def test_reads_equal(sizes):
    e = sphere_amd.Engine(0)
    for n in sizes:
        s = _state(n, n)
        e.load(s.to_state())
        for on in (1, 0, 1):
            e.set_read_staging(on)
            print("read", n, "grains, staging", on, flush=True)
            _same(e.read(), s, n)
    e.close()


def test_reads_from_threads():
    sizes = [500, 18500, 40000, 40000, 90000, 120000]
    states = [_state(n, 7 + k) for k, n in enumerate(sizes)]
    engines = [sphere_amd.Engine(0) for _ in sizes]
    for e, s in zip(engines, states):
        e.load(s.to_state())
    failed = []

    def run(e, s, n):
        try:
            for _ in range(6):
                _same(e.read(), s, n)
        except BaseException as err:
            failed.append((n, err))

    print("reads from", len(sizes), "threads", flush=True)
    threads = [threading.Thread(target=run, args=a) for a in zip(engines, states, sizes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for e in engines:
        e.close()
