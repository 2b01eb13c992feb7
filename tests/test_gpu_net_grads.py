"""Weight and bias gradients of the correction network at the edges of the
weight-gradient tiles (16 x 4 x 4 voxels): grids whose coarse levels are one
voxel wide, partial tiles along each axis, periodic and padded axes, against
the oracle's backward pass; the tolerances are those of the larger grids
(activations whose BF16 rounding ties part the two by a few per cent)."""
import os
import sys

import numpy
import pytest

import sphere_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "oracle"))
import darcy_net as N  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,wrap", [((8, 8, 8), 3), ((8, 40, 24), 2), ((40, 8, 8), 0), ((8, 8, 40), 1)])
def test_gradients_at_tile_edges(shape, wrap):
    import torch
    nz, ny, nx = shape
    rng = numpy.random.default_rng(sum(shape))
    params = N.init_params(rng)
    for w, b in N.split_params(params):
        b[:] = rng.uniform(-0.05, 0.1, b.shape)
    params = params.astype(numpy.float32).astype(numpy.float64)
    inp = rng.standard_normal(shape + (3,)).astype(numpy.float32).astype(numpy.float64)
    R = rng.standard_normal(shape)
    print("net gradients", shape, wrap, flush=True)
    net = sphere_amd.Net(nx, ny, nz, periodic=wrap)
    dev = torch.device("cuda:0")
    p = torch.tensor(params, dtype=torch.float32, device=dev)
    out = torch.empty(nx * ny * nz, dtype=torch.float32, device=dev)
    net.forward(p, torch.tensor(inp.reshape(-1, 3), dtype=torch.float32, device=dev), out)
    g = torch.full((params.size,), 0.5, dtype=torch.float32, device=dev)  # gradients are added
    net.backward(p, torch.tensor(R.ravel(), dtype=torch.float32, device=dev), g)
    torch.cuda.synchronize()
    got = g.cpu().numpy().astype(numpy.float64) - 0.5
    ref = N.backward(N.forward(params, inp, bf16=True, wrap=wrap)[1], R)
    off, rels = 0, []
    for (ci, co), taps in zip(N.LAYERS, N.TAPS_OF):
        for n in (taps * co * ci, co):
            a, b = got[off:off + n], ref[off:off + n]
            off += n
            rels.append(numpy.linalg.norm(a - b) / numpy.linalg.norm(b))
    assert max(rels) <= 8e-2 and numpy.mean(rels) <= 5e-2, rels
    net.close()
