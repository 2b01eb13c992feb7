"""A backward pass adds its gradient to the caller's buffer once: on values of
4096, far above the gradient's own, the result is the rounded sum.  Bound: half
a unit in the last place at 4096 to 8192 (2^-12), and 1e-4 of the largest
gradient for the order in which the blocks' FP32 sums meet (two passes on
zeroed buffers differ by about 1e-6 of it)."""
import numpy
import pytest

import sphere_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,wrap", [(8, 8, 8, 3), (48, 32, 40, 0)])
def test_backward_adds_once(nx, ny, nz, wrap):
    import torch
    rng = numpy.random.default_rng(nx)
    V = nx * ny * nz
    dev = torch.device("cuda:0")
    net = sphere_amd.Net(nx, ny, nz, periodic=wrap)
    n = net.param_count()
    p = torch.tensor(rng.standard_normal(n) * 0.1, dtype=torch.float32, device=dev)
    x = torch.tensor(rng.standard_normal((V, 3)), dtype=torch.float32, device=dev)
    r = torch.tensor(rng.standard_normal(V) / V, dtype=torch.float32, device=dev)
    out = torch.empty(V, dtype=torch.float32, device=dev)
    print("net gradients added to 4096", nx, ny, nz, flush=True)

    def gradient(start):
        g = torch.full((n,), start, dtype=torch.float32, device=dev)
        net.forward(p, x, out)
        net.backward(p, r, g)
        torch.cuda.synchronize()
        return g.cpu().numpy().astype(numpy.float64)

    d, again = gradient(0.0), gradient(0.0)
    big = float(numpy.max(numpy.abs(d)))
    assert 0.0 < big < 1024.0
    assert numpy.max(numpy.abs(d - again)) <= 1e-4 * big  # nothing is left from the pass before
    got = gradient(4096.0)
    assert numpy.max(numpy.abs(got - (4096.0 + d))) <= 2.0 ** -12 + 1e-4 * big
    net.close()
