"""Performance cases of sphere_amd: the work its users have it do.

* ``dem``: an Engine stepping a dense packing (linear or Hertz-Mindlin
  contacts, closed or periodic box under a loaded top wall, bonds),
  then reading the state back, as a run does between two output files.
* ``ensemble``: independent boxes of many sizes stepped together.
* ``darcy``: a packing with a Darcy pore fluid, plain or with the learned
  correction of the pressure solve.
* ``ns``: the Navier-Stokes fluid, alone or moving the grains of an Engine.
* ``net``: the correction network, forward (every learned correction) and
  forward + backward (a training step).

Packings are made on the spot: a periodic tile of grains is pushed to
jamming, repeated over the box and cut to the wanted number of grains, so
that the contacts per grain (about 4.3) and their spread are those of the
grown packings of sphere_amd.workloads.
"""
import numpy
import torch

import sphere_amd
from sphere_amd import _abi, learn

# ----------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------


def listed():
    return [
        # the smallest runs: a closed box of 1,000 grains, where every launch counts
        {"name": "dem_1k", "kind": "dem", "grains": 1000, "tiles": 1, "law": "linear", "closed": True,
         "slots": 32, "bonds": False, "steps": 300},
        # the 10,000 grains of the settling benchmark, settled, in a frictional box
        {"name": "dem_10k", "kind": "dem", "grains": 10000, "tiles": 2, "law": "linear", "closed": True,
         "slots": 32, "bonds": False, "steps": 300},
        # an ordinary shear box: Hertz-Mindlin, bonds, an odd number of grains
        {"name": "shear_87k", "kind": "dem", "grains": 87381, "tiles": 4, "law": "hertz", "closed": False,
         "slots": 32, "bonds": True, "steps": 400},
        # the headline shear box: 1,000,000 lognormal grains, 5% of the contacts bonded
        {"name": "shear_1m", "kind": "dem", "grains": 1000000, "tiles": 11, "law": "hertz",
         "closed": False, "slots": 64, "bonds": True, "steps": 300},
        # a parameter study: 16 independent shear boxes of 5,000 to 60,000 grains
        {"name": "ensemble_16", "kind": "ensemble", "boxes": 16, "grains_min": 5000,
         "grains_max": 60000, "law": "hertz", "steps": 400},
        # a small saturated box on the smallest Darcy grid in use
        {"name": "darcy_8k", "kind": "darcy", "grains": 8000, "tiles": 2, "cells_xy": 16,
         "cells_z": 32, "net": False, "steps": 8},
        # the consolidation benchmark: 200,000 grains on a 48 x 48 x 96 Darcy grid
        {"name": "darcy_200k", "kind": "darcy", "grains": 200000, "tiles": 6, "cells_xy": 48,
         "cells_z": 96, "net": False, "steps": 20},
        # a 32 x 32 x 64 ensemble box with the learned correction in its solves
        {"name": "darcy_learned_59k", "kind": "darcy", "grains": 59332, "tiles": 4, "cells_xy": 32,
         "cells_z": 64, "net": True, "steps": 8},
        # the Navier-Stokes benchmark: a water column of 48 x 48 x 96 cells
        {"name": "ns_column", "kind": "ns", "grains": 0, "tiles": 0, "cells_xy": 48, "cells_z": 96,
         "steps": 2},
        # grains moved by Navier-Stokes water on the grid of their contact search,
        # one fluid solve in ten DEM steps
        {"name": "ns_grains_20k", "kind": "ns", "grains": 20000, "tiles": 2, "cells_xy": 15,
         "cells_z": 44, "steps": 10},
        # one learned correction's network pass on the consolidation grid
        {"name": "net_forward", "kind": "net", "cells_xy": 48, "cells_z": 96, "periodic": 3,
         "backward": False},
        # one training step on the consolidation grid
        {"name": "net_train", "kind": "net", "cells_xy": 48, "cells_z": 96, "periodic": 3,
         "backward": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(float(numpy.exp(rng.uniform(numpy.log(lo), numpy.log(hi))))))


def draw(rng):
    kind = rng.choice(["dem", "dem", "dem", "ensemble", "darcy", "darcy", "ns", "ns", "net", "net"])
    if kind == "dem":
        n = _log_int(rng, 1000, 1000000)
        # 32 x 32 grains across, or fewer in a small box (a tile is about 9.8 across)
        tiles = max(1, int(round((n / 1000.0 / 1.1) ** (1.0 / 3.0) + rng.uniform(-0.3, 0.5))))
        closed = n < 200000 and rng.random() < 0.5
        return {"kind": "dem", "grains": n, "tiles": tiles, "law": rng.choice(["linear", "hertz"]),
                "closed": closed, "slots": rng.choice([32, 64]),
                "bonds": bool(not closed and rng.random() < 0.5),
                "steps": max(100, min(300, int(3e7 / n)))}
    if kind == "ensemble":
        return {"kind": "ensemble", "boxes": rng.randint(2, 16), "grains_min": 5000,
                "grains_max": _log_int(rng, 10000, 60000), "law": rng.choice(["linear", "hertz"]),
                "steps": 200}
    if kind == "darcy":
        net = rng.random() < 0.4
        tiles = rng.randint(2, 6)
        n = tiles * tiles * _log_int(rng, 1200, 5000)
        # the network halves the grid three times; plain solves take any grid
        c = 8 * tiles - (0 if net else rng.randint(0, 3))
        cz = 8 * int(numpy.ceil(n / 900.0 / tiles ** 2 * 1.35 + 1)) + (0 if net else rng.randint(0, 7))
        return {"kind": "darcy", "grains": n, "tiles": tiles, "cells_xy": c, "cells_z": cz, "net": net,
                "steps": rng.randint(3, 8)}
    if kind == "ns":
        if rng.random() < 0.5:
            c = _log_int(rng, 10, 48)
            return {"kind": "ns", "grains": 0, "tiles": 0, "cells_xy": c,
                    "cells_z": rng.randint(c, 2 * c), "steps": 1}
        tiles = rng.randint(1, 2)
        n = tiles * tiles * _log_int(rng, 1000, 4000)
        return {"kind": "ns", "grains": n, "tiles": tiles, "cells_xy": 8 * tiles - rng.randint(0, 1),
                "cells_z": int(numpy.ceil(n / 900.0 / tiles ** 2 * 8 * 1.15)) + rng.randint(3, 9),
                "steps": 10}
    c = 8 * rng.randint(2, 6)
    return {"kind": "net", "cells_xy": c, "cells_z": 8 * rng.randint(max(1, c // 8), c // 4),
            "periodic": rng.choice([0, 1, 3]), "backward": rng.random() < 0.5}


# ----------------------------------------------------------------------
# packings
# ----------------------------------------------------------------------

# Grains of one tile: its edge is then about eight cells of 2.25 mean radii.
TILE_UNIFORM = 900
TILE_LOGNORMAL = 1000
CONTACTS_PER_GRAIN = 4.3


def _tile(seed, lognormal):
    """A periodic cube of grains just past jamming: positions, radii, edge."""
    rng = numpy.random.default_rng(seed)
    m = TILE_LOGNORMAL if lognormal else TILE_UNIFORM
    r = 0.01 * numpy.exp(0.2 * rng.standard_normal(m)) if lognormal else rng.uniform(0.009, 0.011, m)
    r = numpy.clip(r, 0.006, 0.017)
    edge = (numpy.sum(4.0 / 3.0 * numpy.pi * r ** 3) / 0.655) ** (1.0 / 3.0)
    dev = torch.device("cuda:0")
    x = torch.tensor(rng.uniform(0.0, edge, (m, 3)), device=dev)
    rt = torch.tensor(r, device=dev)
    rsum = rt[:, None] + rt[None, :]
    vel = torch.zeros_like(x)

    def gaps(x):
        d = x[:, None, :] - x[None, :, :]
        d -= edge * torch.round(d / edge)
        s = torch.sqrt(torch.sum(d * d, dim=2))
        s.fill_diagonal_(1.0)
        return d, s

    # damped descent of the overlaps, ever closer to the jamming density
    scale = 1.0
    for stage in range(8):
        for _ in range(400):
            d, s = gaps(x)
            over = torch.clamp(scale * rsum - s, min=0.0)
            push = torch.sum((over / s)[:, :, None] * d, dim=1)
            vel = 0.95 * vel + 0.25 * push
            x = x + vel
        d, s = gaps(x)
        ratio = torch.sort((s / rsum).reshape(-1)).values
        want = float(ratio[int(CONTACTS_PER_GRAIN * m)])
        scale = want + (scale - want) * 0.25 if stage < 7 else want
    x = torch.remainder(x, edge).cpu().numpy()
    return x / want, r, edge / want


def _packing(seed, n, tiles, tile, closed):
    """n grains over tiles x tiles copies of a tile, lowest first out of a
    tall stack: positions, radii, box width.  Ordered in layers, rows and
    columns."""
    x0, r0, edge = tile
    m = len(r0)
    rng = numpy.random.default_rng(seed + 1)
    width = edge * tiles
    layers = int(numpy.ceil(n / (m * tiles * tiles) * (1.5 if closed else 1.05))) + 1
    k = numpy.arange(tiles * tiles * layers)
    base = numpy.stack([k % tiles, (k // tiles) % tiles, k // (tiles * tiles)], axis=1) * edge
    x = (base[:, None, :] + x0[None, :, :]).reshape(-1, 3)
    r = numpy.tile(r0, len(k))
    keep = x[:, 2] >= r
    if closed:
        for c in (0, 1):
            keep &= (x[:, c] >= r) & (x[:, c] <= width - r)
    x, r = x[keep], r[keep]
    pick = numpy.argpartition(x[:, 2], n - 1)[:n]
    x, r = x[pick], r[pick]
    cell = (edge ** 3 / m) ** (1.0 / 3.0)
    q = numpy.floor(x / cell).astype(numpy.int64)
    w = int(width / cell) + 2
    order = numpy.argsort((q[:, 2] * w + q[:, 1]) * w + q[:, 0], kind="stable")
    x, r = x[order], r[order]
    x += rng.uniform(-1e-8, 1e-8, x.shape)  # no two tiles quite alike
    x[:, :2] = numpy.clip(x[:, :2], 0.0, width)
    return x, r, width


def _touching(x, r, width, count, rng):
    """`count` of the touching pairs (i < j) that share a cell."""
    cell = 2.05 * float(r.max())
    nx = max(1, int(width / cell))
    q = numpy.minimum((x / (width / nx)).astype(numpy.int64), nx - 1)
    q[:, 2] = (x[:, 2] / (width / nx)).astype(numpy.int64)
    key = (q[:, 2] * nx + q[:, 1]) * nx + q[:, 0]
    order = numpy.argsort(key, kind="stable")
    pairs = []
    for step in range(1, 7):
        i, j = order[:-step], order[step:]
        same = key[i] == key[j]
        i, j = i[same], j[same]
        d = numpy.sqrt(numpy.sum((x[i] - x[j]) ** 2, axis=1))
        hit = d < r[i] + r[j]
        pairs.append(numpy.stack([numpy.minimum(i[hit], j[hit]), numpy.maximum(i[hit], j[hit])], axis=1))
    p = numpy.concatenate(pairs)
    return p[numpy.sort(rng.permutation(len(p))[:count])]


def _box(seed, n, tiles, law, closed, bonds, tile=None):
    """A sim of n grains at small random velocities under a loaded top wall:
    a closed box with frictional walls, or a periodic shear box, its bottom
    layer held and its top layer driven."""
    rng = numpy.random.default_rng(seed + 2)
    x, r, width = _packing(seed, n, tiles, tile or _tile(seed, law == "hertz"), closed)
    top = float(numpy.max(x[:, 2] + r))
    s = sphere_amd.sim(np=n, sid="perf", nw=1)
    s.x[:] = x
    s.radius[:] = r
    s.periodic[0] = 0 if closed else 1
    s.defaultParams(mu_s=0.5, mu_d=0.5, k_n=1.16e7, k_t=1.16e7, gamma_wn=1e2, gamma_wt=1e2)
    s.mu_ws = numpy.array([0.5])
    s.mu_wd = numpy.array([0.5])
    s.g[:] = [0.0, 0.0, -9.81]
    s.gamma_n[0] = 2e2 if law == "hertz" else 5e2
    r_max = float(r.max())
    if law == "hertz":
        s.contactmodel[0] = 3
        s.setYoungsModulus(7e9)
        s.setPoissonsRatio(0.3)
        stiff = numpy.pi / 2.0 * 7e9 * r_max
    else:
        s.contactmodel[0] = 2
        stiff = 1.16e7
    s.defineWorldBoundaries(L=[width, width, top + 4.0 * r_max], dx=2.31 * r_max)
    m_min = 2600.0 * 4.0 / 3.0 * numpy.pi * float(r.min()) ** 3
    dt = 0.17 * numpy.sqrt(m_min / stiff)
    s.vel[:] = rng.uniform(-1e-2, 1e-2, (n, 3))
    s.angvel[:] = rng.uniform(-1.0, 1.0, (n, 3))
    s.w_n[0, :] = [0.0, 0.0, -1.0]
    s.w_x[0] = top
    s.wmode[0] = 1
    s.w_m[0] = s.totalMass()
    s.w_sigma0[0] = 10e3 if law == "hertz" else 50e3
    if not closed:
        s.fixvel[x[:, 2] < 2.0 * r_max] = 1.0
        s.vel[s.fixvel > 0.0, :] = 0.0
        high = x[:, 2] > top - 2.0 * r_max
        s.fixvel[high] = 1.0
        s.vel[high, 0], s.vel[high, 1] = 0.01, 0.0
        s.angvel[s.fixvel > 0.0, :] = 0.0
    if bonds:
        nb = n // 10
        p = _touching(x, r, width, nb, rng)
        s.lambda_bar[0] = 1.0
        s.bonds = p.astype(numpy.uint32)
        s.bonds_delta_n, s.bonds_omega_n = numpy.zeros(nb), numpy.zeros(nb)
        s.bonds_delta_t, s.bonds_omega_t = numpy.zeros((nb, 3)), numpy.zeros((nb, 3))
        s.nb0 = numpy.ones(1, dtype=numpy.uint32) * nb
    _endless(s, dt)
    return s


def _endless(s, dt):
    """Times of a run whose next output lies beyond every step taken here."""
    s.time_dt[0] = dt
    s.time_current[0] = 0.0
    s.time_total[0] = 9.0
    s.time_file_dt[0] = 9.0
    s.time_step_count[0] = 0


def _saturated(seed, n, tiles, cells_xy, cells_z):
    """The consolidation box: a periodic packing under a 20 kPa wall, its
    grid the Darcy grid (fluid as in workloads.consolidation_finish)."""
    rng = numpy.random.default_rng(seed + 2)
    x, r, width = _packing(seed, n, tiles, _tile(seed, False), False)
    top = float(numpy.max(x[:, 2] + r))
    s = sphere_amd.sim(np=n, sid="perf", nw=1)
    s.x[:] = x
    s.radius[:] = r
    s.periodic[0] = 1
    s.contactmodel[0] = 2
    s.defaultParams(mu_s=0.5, mu_d=0.5, k_n=1.16e7, k_t=1.16e7, gamma_n=5e2, gamma_wn=1e2,
                    gamma_wt=0.0)
    s.g[:] = [0.0, 0.0, -9.81]
    cell = width / cells_xy
    s.num = numpy.array([cells_xy, cells_xy, cells_z], dtype=numpy.uint32)
    s.L = numpy.array([width, width, max(cells_z * cell, top * 1.05)])
    s.vel[:] = rng.uniform(-1e-3, 1e-3, (n, 3))
    s.w_n[0, :] = [0.0, 0.0, -1.0]
    s.w_x[0] = top
    s.wmode[0] = 1
    s.w_m[0] = s.totalMass()
    s.w_sigma0[0] = 200e3
    m_min = 2600.0 * 4.0 / 3.0 * numpy.pi * float(r.min()) ** 3
    _endless(s, 0.17 * numpy.sqrt(m_min / 1.16e9))
    return s


def _darcy(s):
    s.initFluid(mu=1.04e-7, rho=1000.0, p=0.0, cfd_solver=1)
    s.setFluidCompressibility(1.43e-8)
    s.setPermeabilityPrefactor(3.5e-13, verbose=False)
    s.setFluidBottomNoFlow()
    s.setFluidTopFixedPressure()
    s.setTolerance(1e-8)
    s.setMaxIterations(200000)
    s.setDEMstepsPerCFDstep(1)


# ----------------------------------------------------------------------
# prepare and run
# ----------------------------------------------------------------------


def _engine(s, slots=32):
    e = sphere_amd.Engine(0, nc=slots)
    e.load(s.to_state())
    return e


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dem":
        s = _box(seed, case["grains"], case["tiles"], case["law"], case["closed"], case["bonds"])
        return {"case": case, "engine": _engine(s, case["slots"])}
    if kind == "ensemble":
        rng = numpy.random.default_rng(1000 * case["boxes"] + case["grains_max"])
        lo, hi = numpy.log(case["grains_min"]), numpy.log(case["grains_max"])
        tile = _tile(seed, case["law"] == "hertz")
        engines = []
        for b, n in enumerate(numpy.exp(rng.uniform(lo, hi, case["boxes"]))):
            s = _box(seed + 100 * b, int(n), 2 if n < 20000 else 3, case["law"], False, False, tile)
            s.mu_s[0] = s.mu_d[0] = rng.uniform(0.3, 0.7)
            s.w_sigma0[0] = rng.uniform(5e3, 80e3)
            s.vel[s.vel[:, 0] == 0.01, 0] = rng.uniform(1e-3, 1e-1)
            engines.append(_engine(s, 64))
        return {"case": case, "engines": engines, "ensemble": sphere_amd.Ensemble(engines)}
    if kind == "darcy":
        s = _saturated(seed, case["grains"], case["tiles"], case["cells_xy"], case["cells_z"])
        _darcy(s)
        e = _engine(s)
        if case["net"]:
            e.set_darcy_net(learn.init_params(seed), 8)
        return {"case": case, "engine": e}
    if kind == "ns":
        return _prepare_ns(case, seed)
    nx, nz = case["cells_xy"], case["cells_z"]
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(seed)
    V = nx * nx * nz
    # a normalized residual (waves and noise), the cell coupling log(1 + D) and
    # a held top layer; the loss's derivative where the target follows the waves
    z, y, x = torch.meshgrid(torch.arange(nz), torch.arange(nx), torch.arange(nx), indexing="ij")
    wave = torch.zeros((nz, nx, nx))
    for k in torch.rand((6, 4), generator=g):
        wave += torch.cos(6.2832 * ((3 * k[0]).round() * x / nx + (3 * k[1]).round() * y / nx
                                    + 2.0 * k[2] * z / nz + k[3]))
    wave = (wave / 6.0).reshape(V)
    inp = torch.empty((V, 3))
    inp[:, 0] = 0.8 * wave + 0.2 * torch.rand(V, generator=g)
    inp[:, 1] = 0.5 + torch.rand(V, generator=g)
    inp[:, 2] = (torch.arange(V) >= V - 2 * nx * nx).float()
    grad = -(wave + 0.2 * torch.rand(V, generator=g)) * (2.0 / V)
    params = torch.from_numpy(learn.init_params(seed)).to(dev)
    return {"case": case, "net": sphere_amd.Net(nx, nx, nz, periodic=case["periodic"]),
            "params": params, "inp": inp.to(dev), "grad": grad.to(dev),
            "out": torch.empty(V, device=dev)}


def _prepare_ns(case, seed):
    rng = numpy.random.default_rng(seed)
    c, nz = case["cells_xy"], case["cells_z"]
    if case["grains"]:
        s = _saturated(seed, case["grains"], case["tiles"], c, nz)
        s.wmode[0] = 0
        # the linear law's own time step; the Darcy boxes need a shorter one
        s.time_dt[0] *= 10.0
        L, dt, ndem = [float(v) for v in s.L], float(s.time_dt[0]), 10
        v = numpy.zeros((c, c, nz, 3))
    else:
        cell = 0.0231
        L, dt, ndem = [c * cell, c * cell, nz * cell], 1e-4, 1
        v = 0.01 * rng.standard_normal((c, c, nz, 3))
    dz = L[2] / nz
    p = numpy.broadcast_to(1000.0 * 9.81 * dz * (nz - 1 - numpy.arange(nz)), (c, c, nz)).copy()
    P = _abi.ns_params(c, c, nz, L, dt, mu=8.9e-4, rho_f=1000.0, g=(0.0, 0.0, -9.81), bc_bot=1, bc_top=0,
                       tolerance=1.0e-8, maxiter=10000, ndem=ndem)
    fluid = sphere_amd.NavierStokes(P, v, p)
    engine = None
    if case["grains"]:
        engine = _engine(s)
        engine.attach_fluid(fluid)
    else:
        fluid.step(12)  # past the first, long solve from rest: water in motion
    return {"case": case, "engine": engine, "fluid": fluid}


def _state_of(engine):
    a = engine.read().arrays
    return {k: a[k] for k in sorted(a) if k not in ("color", "p_constant", "bonds") and a[k].size > 3}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dem" or kind == "darcy":
        state["engine"].step(case["steps"])
        return _state_of(state["engine"])
    if kind == "ensemble":
        state["ensemble"].step(case["steps"])
        got = [e.read() for e in state["engines"]]
        return {k: [b.arrays[k] for b in got] for k in ("x", "vel", "angvel")}
    if kind == "ns":
        out = {}
        if state["engine"] is not None:
            state["engine"].step(case["steps"])
            out["grains"] = _state_of(state["engine"])
        else:
            state["fluid"].step(case["steps"])
        out["v"], out["p"], out["phi"], _ = state["fluid"].read()
        return out
    state["net"].forward(state["params"], state["inp"], state["out"])
    if not case["backward"]:
        return state["out"]
    g = torch.zeros_like(state["params"])
    state["net"].backward(state["params"], state["grad"], g)
    return {"out": state["out"], "grad": g}


# ----------------------------------------------------------------------
# work, tolerance, exact
# ----------------------------------------------------------------------

# Bytes of a grain's state in a read, and what one step must move: per grain
# x, vel, angvel, angpos, xyzsum and both previous accelerations in and out,
# es and ev in and out, force, torque, es_dot, ev_dot, p and the wall force
# out; per contact the partner and the tangential spring in and out.
GRAIN_READ = 28 * 8
GRAIN_STEP = 480
CONTACT_STEP = 52
NET_LAYERS = [(3, 16, 1), (16, 32, 8), (32, 48, 64), (48, 64, 512), (64, 48, 512), (48, 32, 64),
              (32, 16, 8), (16, 16, 1)]


def _dem_work(n, steps, read=GRAIN_READ):
    z = CONTACTS_PER_GRAIN
    return {"bytes": n * (steps * (GRAIN_STEP + CONTACT_STEP * z) + read),
            "flops": n * steps * (250.0 + 200.0 * z)}


def work(case):
    kind = case["kind"]
    if kind == "dem":
        return _dem_work(case["grains"], case["steps"])
    if kind == "ensemble":
        lo, hi = case["grains_min"], case["grains_max"]
        n = case["boxes"] * (hi - lo) / numpy.log(hi / lo)  # the mean of a log-uniform size
        return _dem_work(n, case["steps"], 11 * 8)
    if kind == "net":
        V = case["cells_xy"] ** 2 * case["cells_z"]
        flops = sum(2.0 * 27 * ci * co * V / f for ci, co, f in NET_LAYERS) + 2.0 * 16 * V
        params = 4 * sum(27 * ci * co + co for ci, co, _ in NET_LAYERS)
        if case["backward"]:
            return {"bytes": V * 20.0 + 2 * params, "flops": 3.0 * flops}
        return {"bytes": V * 16.0 + params, "flops": flops}
    cells = case["cells_xy"] ** 2 * case["cells_z"]
    n = case["grains"]
    grains = _dem_work(n, case["steps"])
    # fields in and out once, and per iteration of the pressure p in and out
    # and the cell's constants; the counts are those of ordinary solves
    if kind == "darcy":
        sweeps, flops = 400.0, 45.0
        w = {"bytes": cells * case["steps"] * (120.0 + 40.0 * sweeps),
             "flops": cells * case["steps"] * flops * sweeps}
    else:
        # (the long solves of moving grains end at the iteration limit)
        solves = case["steps"] / (10 if n else 1)
        its = min(10000.0, 6000.0 * (case["cells_z"] / 96.0) ** 2) if n == 0 else 10000.0
        w = {"bytes": cells * solves * (200.0 + 48.0 * its), "flops": cells * solves * 30.0 * its}
    return {k: w[k] + grains[k] for k in w}


def tolerance(case):
    # Measured with the grains renumbered, so that every sum over contacts and
    # cells runs in another order: up to 2e-10 and 9e-9 after 300 steps (linear
    # contacts slip at slightly other times, and each step carries that on),
    # 1e-10 and 1.4e-9 in the solved pressures.  The network's activations are
    # bf16: against 64 bits its output is about 0.5% off.
    if case["kind"] == "net":
        return {"rel": 0.02, "max": 0.5}
    return {"rel": 1e-8, "max": 1e-6}


def _small(case):
    return case["grains"] <= 2500 and not case["bonds"]


def exact(case, seed):
    if case["kind"] == "net":
        return _exact_net(case, seed)
    if case["kind"] == "dem" and _small(case):
        return _exact_dem(case, seed)
    return None  # hundreds of steps or thousands of sweeps: minutes in plain torch


def _exact_net(case, seed):
    """The correction network in 64 bits: 3x3x3 convolutions as sums of 27
    shifted products, ReLU, average pooling, nearest upsampling with the skip
    added, a pointwise head."""
    st = prepare(case, seed)
    n, nz, per = case["cells_xy"], case["cells_z"], case["periodic"]
    params = st["params"].double().requires_grad_(case["backward"])

    def conv(a, w, b):
        # a [z, y, x, ci]; w [27, co, ci], tap = (dz * 3 + dy) * 3 + dx
        def pad(t, dim, wrap):
            if wrap:
                return torch.cat([t.narrow(dim, t.shape[dim] - 1, 1), t, t.narrow(dim, 0, 1)], dim)
            z = torch.zeros_like(t.narrow(dim, 0, 1))
            return torch.cat([z, t, z], dim)
        q = pad(pad(pad(a, 2, per & 1), 1, per & 2), 0, 0)
        dz, dy, dx, ci = a.shape
        out = torch.zeros((dz * dy * dx, w.shape[1]), dtype=torch.float64, device=a.device) + b
        for t in range(27):
            k, j, i = t // 9, (t // 3) % 3, t % 3
            part = q[k:k + dz, j:j + dy, i:i + dx].reshape(-1, ci)
            out = out + torch.matmul(part, w[t].t().contiguous())
        return out.reshape(dz, dy, dx, -1)

    def pool(a):
        z, y, x, c = a.shape
        return a.reshape(z // 2, 2, y // 2, 2, x // 2, 2, c).mean(dim=(1, 3, 5))

    def up(a):
        z, y, x, c = a.shape
        return a[:, None, :, None, :, None].expand(z, 2, y, 2, x, 2, c).reshape(2 * z, 2 * y, 2 * x, c)

    layers, o = [], 0
    for ci, co, taps in learn.LAYERS:
        w = params[o:o + taps * co * ci].reshape(taps, co, ci)
        o += taps * co * ci
        layers.append((w, params[o:o + co]))
        o += co
    a0 = st["inp"].double().reshape(nz, n, n, 3)
    a1 = torch.relu(conv(a0, *layers[0]))
    a2 = torch.relu(conv(pool(a1), *layers[1]))
    a3 = torch.relu(conv(pool(a2), *layers[2]))
    a4 = torch.relu(conv(pool(a3), *layers[3]))
    u3 = up(torch.relu(conv(a4, *layers[4]))) + a3
    u2 = up(torch.relu(conv(u3, *layers[5]))) + a2
    u1 = up(torch.relu(conv(u2, *layers[6]))) + a1
    y = torch.relu(conv(u1, *layers[7])).reshape(-1, 16)
    out = (y * layers[8][0][0, 0]).sum(dim=1) + layers[8][1]
    if not case["backward"]:
        return out
    (out * st["grad"].double()).sum().backward()
    return {"out": out.detach(), "grad": params.grad}


def _exact_dem(case, seed):
    """The same steps with every pair tested: overlaps of the nearest images,
    the contact and wall laws with their tangential springs, the third-order
    Taylor update."""
    s = _box(seed, case["grains"], case["tiles"], case["law"], case["closed"], False)
    dev = torch.device("cuda:0")

    def on(a):
        return torch.tensor(numpy.ascontiguousarray(a), dtype=torch.float64, device=dev)

    n, dt, rho = case["grains"], float(s.time_dt[0]), float(s.rho[0])
    x, v, w, r = on(s.x), on(s.vel), on(s.angvel), on(s.radius)
    fix = on(s.fixvel)
    L = [float(t) for t in s.L]
    k_n, k_t, E = float(s.k_n[0]), float(s.k_t[0]), float(s.E[0])
    g_n, g_wn, g_wt = float(s.gamma_n[0]), float(s.gamma_wn[0]), float(s.gamma_wt[0])
    g_t, mu_s, mu_d, mu_wd = float(s.gamma_t[0]), float(s.mu_s[0]), float(s.mu_d[0]), float(s.mu_wd[0])
    grav = on(s.g)
    closed, hertz = case["closed"], case["law"] == "hertz"
    wall = [float(s.w_x[0]), 0.0, 0.0, float(s.w_m[0]), float(s.w_sigma0[0])]
    spring = torch.zeros((n, n, 3), dtype=torch.float64, device=dev)
    acc0, ang0 = torch.zeros_like(x), torch.zeros_like(x)
    angpos, moved = torch.zeros_like(x), torch.zeros_like(x)
    es, ev = torch.zeros_like(r), torch.zeros_like(r)
    mass = 4.0 / 3.0 * numpy.pi * r ** 3 * rho
    inertia = 0.4 * mass * r * r
    rs = r[:, None] + r[None, :]
    if hertz:
        nu = float(s.k_r[0])
        R = torch.sqrt(r[:, None] * r[None, :] / rs)
        kn_h = 4.0 / 3.0 * E / (2.0 * (1.0 - nu * nu)) * R
        kt_h = 8.0 * (E / (2.0 * (1.0 + nu))) / (2.0 * (2.0 - nu)) * R

    def length(a):
        return torch.sqrt(torch.sum(a * a, dim=-1))

    def over(a, b):
        return torch.where(b > 0.0, a / torch.where(b > 0.0, b, torch.ones_like(b)), torch.zeros_like(a))

    for step in range(case["steps"]):
        d = x[:, None, :] - x[None, :, :]
        if not closed:
            for c in (0, 1):
                d[..., c] -= L[c] * torch.round(d[..., c] / L[c])
        dist = length(d)
        dist.fill_diagonal_(1e9)
        I, J = torch.nonzero(dist < rs, as_tuple=True)
        l, rsum = dist[I, J], rs[I, J]
        delta = l - rsum
        nrm = d[I, J] / l[:, None]
        arm_i, arm_j = (r[I] + delta / 2.0)[:, None], (r[J] + delta / 2.0)[:, None]
        vl = v[I] - v[J]
        vc = vl + arm_i * torch.linalg.cross(nrm, w[I]) + arm_j * torch.linalg.cross(nrm, w[J])
        vn = torch.sum(vl * nrm, dim=1)
        vt = vc - torch.sum(vc * nrm, dim=1, keepdim=True) * nrm
        vt_l = length(vt)
        old = spring[I, J]
        old = old - torch.sum(old * nrm, dim=1, keepdim=True) * nrm
        if hertz:
            sd = torch.sqrt(-delta)
            qd = torch.sqrt(sd)
            kn, kt = kn_h[I, J], kt_h[I, J]
            fn = torch.clamp(kn * -delta * sd - g_n * qd * vn, min=0.0)
            e_v = g_n * vn * vn
            ft = -(kt * sd)[:, None] * old - (g_t * qd)[:, None] * vt
            lim = torch.where(vt_l > float(numpy.float32(0.001)), mu_d, mu_s) * fn
            ft_l = length(ft)
            slip = ft_l > lim
            ft = torch.where(slip[:, None], over(lim, ft_l)[:, None] * ft, ft)
            new = torch.where(slip[:, None], (ft + (g_t * qd)[:, None] * vt) / -(kt * sd)[:, None],
                              old + dt * vt)
            e_s = torch.where(slip, length(old - new) * kt / dt, 0.0)
        else:
            fn = torch.clamp(-k_n * delta - g_n * vn, min=0.0)
            e_v = 0.5 * g_n * vn * vn + 0.5 * g_t * vt_l * vt_l
            new = old + dt * vt
            ft = -k_t * new - g_t * vt
            lim = mu_s * fn
            ft_l = length(ft)
            slip = ft_l > lim
            t = over(ft, ft_l[:, None].expand_as(ft))
            ft = torch.where(slip[:, None], lim[:, None] * t, ft)
            new = torch.where(slip[:, None], -(mu_d * fn[:, None] * t + g_t * vt) / k_t, new)
            e_s = torch.where(slip, 0.5 * length(ft) * vt_l, 0.0)
        spring = torch.zeros_like(spring)
        spring[I, J] = new
        pair_f = fn[:, None] * nrm + ft
        pair_t = torch.linalg.cross(-arm_i * nrm, ft)
        F = torch.zeros_like(x).index_add_(0, I, pair_f)
        T = torch.zeros_like(x).index_add_(0, I, pair_t)
        press = torch.zeros_like(r).index_add_(0, I, fn / (4.0 * numpy.pi * r[I] ** 2))
        ev_dot = torch.zeros_like(r).index_add_(0, I, e_v)
        es_dot = torch.zeros_like(r).index_add_(0, I, e_s)
        planes = [([0.0, 0.0, -1.0], wall[0], wall[1]), ([0.0, 0.0, 1.0], 0.0, 0.0)]
        if closed:
            planes += [([-1.0, 0.0, 0.0], L[0], 0.0), ([1.0, 0.0, 0.0], 0.0, 0.0),
                       ([0.0, -1.0, 0.0], L[1], 0.0), ([0.0, 1.0, 0.0], 0.0, 0.0)]
        wall_f = 0.0
        for k, (normal, at, speed) in enumerate(planes):
            axis = [abs(c) for c in normal].index(1.0)
            q = x[:, axis]
            delta = at - (q + r) if normal[axis] < 0.0 else q - r - at
            hit = delta < 0.0
            nv = on(normal)
            vc = v + (r + delta / 2.0)[:, None] * torch.linalg.cross(nv.expand_as(w), w) + speed
            vn = torch.sum(v * nv, dim=1)
            vt = vc - torch.sum(vc * nv, dim=1, keepdim=True) * nv
            vt_l = length(vt)
            kw = numpy.pi / 2.0 * E * r if E > 0.001 else k_n
            fn = torch.where(hit, torch.clamp(-kw * delta - g_wn * vn, min=0.0), 0.0)
            lim = mu_wd * fn
            visc = g_wt * vt_l
            slip = hit & (visc >= lim) & (vt_l > 0.0) & (g_wt > 0.0)
            ft = torch.where(slip, -over(lim, vt_l), torch.where(hit, -g_wt, 0.0))[:, None] * vt
            f = fn[:, None] * nv
            F = F + (f + ft)
            T = T + torch.linalg.cross(-(r + delta * 0.5)[:, None] * nv, ft)
            press = press + fn / (4.0 * numpy.pi * r * r)
            ev_dot = ev_dot + torch.where(hit, g_wn * vn * vn, 0.0)
            es_dot = es_dot + torch.where(slip, length(ft) * vt_l, 0.0)
            if k == 0:
                wall_f = float(torch.sum(f * nv))
        es, ev = es + es_dot * dt, ev + ev_dot * dt
        acc = F / mass[:, None] + grav
        ang = T / inertia[:, None]
        held = fix > 0.0001
        acc[held, 0] = acc[held, 1] = 0.0
        acc[held, 2] -= grav[2]
        ang[held] = 0.0
        jerk, angjerk = (acc - acc0) / dt, (ang - ang0) / dt
        dx = v * dt + 0.5 * acc * dt ** 2 + jerk * dt ** 3 / 6.0
        angpos = angpos + w * dt + 0.5 * ang * dt ** 2 + angjerk * dt ** 3 / 6.0
        x, moved = x + dx, moved + dx
        v = v + acc * dt + 0.5 * jerk * dt ** 2
        w = w + ang * dt + 0.5 * angjerk * dt ** 2
        acc0, ang0 = acc, ang
        if not closed:
            for c in (0, 1):
                x[:, c] = torch.where(x[:, c] < 0.0, x[:, c] + L[c], x[:, c])
                x[:, c] = torch.where(x[:, c] > L[c], x[:, c] - L[c], x[:, c])
        a = (wall_f - wall[4] * L[0] * L[1]) / wall[3]
        j = (a - wall[2]) / dt
        wall[0] += wall[1] * dt + 0.5 * a * dt ** 2 + j * dt ** 3 / 6.0
        wall[1] += a * dt + 0.5 * j * dt ** 2
        wall[2] = a

    def four(a, last):
        return torch.cat([a, last[:, None]], dim=1).reshape(-1)

    return {"x": four(x, r), "vel": four(v, fix), "angvel": w.reshape(-1), "angpos": angpos.reshape(-1),
            "xyzsum": moved.reshape(-1), "force": F.reshape(-1), "torque": T.reshape(-1), "p": press,
            "es": es, "ev": ev, "es_dot": es_dot, "ev_dot": ev_dot}
