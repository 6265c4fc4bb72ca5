"""The work a program built on this library has it do, as measurable cases.

Each case is one pass over a piece of an immersed-boundary time step (or of a
regrid) through the library's public Python layer:

  ib      spread the force, fill the velocity's periodic ghosts, interpolate at
          the same positions, advance the positions (one periodic patch, 2-D or
          3-D, every kernel width, FP64 and FP32C); points binned beforehand, as
          IBAMR associates points with patches at a regrid only
  amr     the same on a fine level of many patches of unequal sizes, with the
          same-level ghost fill
  walls   a closed box cut into patches: spread, fold of the ghost forces at the
          walls, wall ghost values of the velocity, interpolation
  step    a captured time step of several structures with two delta kernels,
          points binned every step
  regrid  redistribution of the points over the patches, permutation of their
          data, binning
  forces  springs, beams and target points of closed rings
  fe      quadrature points of a hexahedral or quadrilateral mesh, spread and
          interpolation there, the nodal right-hand side

Sizes are those of the repository's tests and benchmark or generic ones; draw()
spreads them over the same ranges.
"""
import math

import numpy as np
import torch

import ibamr_amd as ia
from ibamr_amd import fe, ibstep, structure

DEV = "cuda"
WIDTH = {"PIECEWISE_LINEAR": 2, "BSPLINE_3": 3, "IB_4": 4, "IB_6": 6}
GHOST = {"PIECEWISE_LINEAR": 2, "BSPLINE_3": 3, "IB_4": 3, "IB_6": 4}


# --------------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest use: a 2-D elastic membrane on 128^2, the classic first example
        {"name": "membrane_2d_128", "kind": "ib", "ndim": 2, "n": 128, "kernel": "IB_4", "prec": "fp64",
         "points": 1024, "layout": "shell", "order": "regrid", "tune": False},
        # a thick 2-D structure on a fine grid whose size is no multiple of a tile
        {"name": "disc_2d_1000", "kind": "ib", "ndim": 2, "n": 1000, "kernel": "IB_4", "prec": "fp64",
         "points": 200000, "layout": "solid", "order": "regrid", "tune": False},
        # a small 3-D run (a coarse trial run, or one rank's share): launches and tails count
        {"name": "small_3d_40", "kind": "ib", "ndim": 3, "n": 40, "kernel": "IB_4", "prec": "fp64",
         "points": 3000, "layout": "uniform", "order": "generated", "tune": False},
        # an ordinary 3-D run in double precision: a shell on 256^3
        {"name": "sphere_256_fp64", "kind": "ib", "ndim": 3, "n": 256, "kernel": "IB_4", "prec": "fp64",
         "points": 1 << 20, "layout": "shell", "order": "regrid", "tune": False},
        # the largest single-patch run, FP32 grid data with compensated sums (the benchmark's workload)
        {"name": "mixed_512_fp32c", "kind": "ib", "ndim": 3, "n": 512, "kernel": "IB_6", "prec": "fp32c",
         "points": 1 << 23, "layout": "mixed", "order": "regrid", "tune": True},
        # the same in double precision, the reference's own form
        {"name": "mixed_512_fp64", "kind": "ib", "ndim": 3, "n": 512, "kernel": "IB_6", "prec": "fp64",
         "points": 1 << 23, "layout": "mixed", "order": "regrid", "tune": False},
        # a refined level of many patches around thin shells
        {"name": "amr_512_fp32c", "kind": "amr", "n": 512, "kernel": "BSPLINE_3", "prec": "fp32c",
         "points": 1 << 21, "shells": 4, "tune": True},
        # a whole captured step of 64 shells of two kernels, binned every step
        {"name": "step_384_fp32c", "kind": "step", "n": 384, "prec": "fp32c", "shells": 64, "points": 2700000},
        # a closed box (a driven cavity or a channel with walls) cut into patches
        {"name": "walls_160_fp64", "kind": "walls", "nx": 160, "ny": 144, "nz": 200, "cuts": 2, "kernel": "IB_4",
         "prec": "fp64", "centering": "side", "depth": 1, "points": 300000},
        # a regrid of two million points over 27 patches
        {"name": "regrid_256", "kind": "regrid", "n": 256, "cuts": 3, "prec": "fp64", "points": 1 << 21},
        # force generation of closed rings with bending and target points
        {"name": "rings_forces", "kind": "forces", "prec": "fp64", "nodes": 1500000, "rings": 64, "every": 4},
        # a solid finite-element body: HEX8 elements with 2^3 quadrature points
        {"name": "solid_fe_256", "kind": "fe", "ndim": 3, "n": 256, "kernel": "IB_4", "prec": "fp64", "edge": 48,
         "rule": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ib2", "ib3", "ib3", "ib3", "amr", "step", "walls", "regrid", "forces", "fe"])
    prec = rng.choice(["fp64", "fp32c"])
    kernel = rng.choice(["IB_4", "IB_6", "BSPLINE_3", "PIECEWISE_LINEAR"])
    if kind == "ib2":
        n = _log(rng, 40, 1400)
        return {"kind": "ib", "ndim": 2, "n": n, "kernel": kernel, "prec": prec, "points": _log(rng, 500, 400000),
                "layout": rng.choice(["uniform", "shell", "solid", "mixed"]),
                "order": rng.choice(["regrid", "generated"]), "tune": False}
    if kind == "ib3":
        n = _log(rng, 33, 440)
        return {"kind": "ib", "ndim": 3, "n": n, "kernel": kernel, "prec": prec,
                "points": _log(rng, 2000, min(4000000, n ** 3)),
                "layout": rng.choice(["uniform", "shell", "solid", "mixed"]),
                "order": rng.choice(["regrid", "generated"]), "tune": rng.choice([False, True])}
    if kind == "amr":
        return {"kind": "amr", "n": 64 * rng.randint(3, 8), "kernel": kernel, "prec": prec,
                "points": _log(rng, 50000, 1500000), "shells": rng.randint(1, 4), "tune": rng.choice([False, True])}
    if kind == "step":
        return {"kind": "step", "n": rng.randint(64, 320), "prec": prec, "shells": rng.randint(2, 48),
                "points": _log(rng, 20000, 2000000)}
    if kind == "walls":
        side = rng.random() < 0.6
        return {"kind": "walls", "nx": rng.randint(40, 180), "ny": rng.randint(40, 180), "nz": rng.randint(40, 180),
                "cuts": rng.randint(1, 2), "kernel": kernel, "prec": prec, "centering": "side" if side else "cell",
                "depth": 1 if side else rng.randint(1, 3), "points": _log(rng, 5000, 400000)}
    if kind == "regrid":
        return {"kind": "regrid", "n": rng.randint(60, 400), "cuts": rng.randint(1, 4), "prec": prec,
                "points": _log(rng, 20000, 4000000)}
    if kind == "forces":
        return {"kind": "forces", "prec": prec, "nodes": _log(rng, 2000, 1500000), "rings": rng.randint(1, 100),
                "every": rng.randint(2, 20)}
    nd = rng.choice([2, 3])
    return {"kind": "fe", "ndim": nd, "n": rng.randint(64, 900) if nd == 2 else rng.randint(64, 300),
            "kernel": kernel, "prec": prec, "edge": _log(rng, 20, 250) if nd == 2 else _log(rng, 8, 48),
            "rule": rng.randint(2, 3)}


# --------------------------------------------------------------------------- inputs

def _dtype(prec):
    return torch.float64 if prec == "fp64" else torch.float32


def _prec(prec):
    return ia.FP64 if prec == "fp64" else ia.FP32C


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float64)


def _directions(g, n, ndim):
    d = _randn(g, n, ndim)
    return d / d.norm(dim=1, keepdim=True)


def _points(g, n, ndim, h, layout):
    """n positions in the unit box: uniform, a shell of radius 0.3 and thickness
    2h, a solid ball of radius 0.3, or half uniform and half shell."""
    if layout == "mixed":
        return torch.cat([_points(g, n // 2, ndim, h, "uniform"), _points(g, n - n // 2, ndim, h, "shell")])
    if layout == "uniform":
        return _rand(g, n, ndim)
    d = _directions(g, n, ndim)
    if layout == "shell":
        return 0.5 + (0.3 - h + 2 * h * _rand(g, n, 1)) * d
    return 0.5 + 0.3 * _rand(g, n, 1) ** (1.0 / ndim) * d


def _cells(X, h):
    return torch.floor(X / h).long()


def _regrid_order(X, h, n):
    """The points by cell (x fastest), the order local data has after a regrid."""
    c = _cells(X, h)
    key = torch.zeros(X.shape[0], dtype=torch.int64, device=DEV)
    for d in reversed(range(X.shape[1])):
        key = key * n + c[:, d]
    return X[torch.argsort(key, stable=True)].contiguous()


def _pool(shapes, dtype, g=None):
    """One allocation holding arrays of the given shapes (values uniform in
    [-1, 1) from g, or zeros), and views of them."""
    sizes = [int(np.prod(s)) for s in shapes]
    if g is None:
        flat = torch.zeros(sum(sizes), dtype=dtype, device=DEV)
    else:
        flat = (2 * _rand(g, sum(sizes)) - 1).to(dtype)
    return flat, [v.view(s) for v, s in zip(torch.split(flat, sizes), shapes)]


def _shapes(level, gcw, centering, depth=1):
    return [ia.array_shape(level, p, gcw, centering, axis=a, depth=depth)
            for p in range(len(level.patches)) for a in range(level.ndim if centering == ia.SIDE else 1)]


def _ib_inputs(c, seed):
    nd, n = c["ndim"], c["n"]
    h = 1.0 / n
    g = _gen(seed)
    X = _points(g, c["points"], nd, h, c["layout"])
    if c["order"] == "regrid":
        X = _regrid_order(X, h, n)
    F = _randn(g, c["points"], nd).to(_dtype(c["prec"]))
    level = ia.Level.uniform_periodic(n, nd)
    gcw = [GHOST[c["kernel"]]] * nd
    flat, u = _pool(_shapes(level, gcw, ia.SIDE), _dtype(c["prec"]), g)
    return level, gcw, X, F, u


def _amr_geometry(c):
    """A fine level around c["shells"] spheres: the domain cut along each axis
    into edges from {16, 32, 48, 64} (a fixed pattern), the bricks the shells'
    points can reach kept as patches."""
    n = c["n"]
    h = 1.0 / n
    pattern = [[64, 48, 16, 64, 32, 32], [48, 64, 32, 16, 64, 32], [32, 64, 64, 48, 16, 32]]
    cuts = []
    for p in pattern:
        e, k = [0], 0
        while e[-1] < n:
            e.append(min(n, e[-1] + p[k % len(p)]))
            k += 1
        cuts.append(e)
    spheres = [((0.32, 0.35, 0.36), 0.17), ((0.66, 0.6, 0.34), 0.15), ((0.4, 0.64, 0.68), 0.13),
               ((0.7, 0.28, 0.7), 0.11)][:c["shells"]]
    patches = []
    for k in range(len(cuts[2]) - 1):
        for j in range(len(cuts[1]) - 1):
            for i in range(len(cuts[0]) - 1):
                lo = [cuts[0][i], cuts[1][j], cuts[2][k]]
                hi = [cuts[0][i + 1] - 1, cuts[1][j + 1] - 1, cuts[2][k + 1] - 1]
                for ctr, r in spheres:
                    near = math.sqrt(sum(max(lo[d] * h - ctr[d], 0.0, ctr[d] - (hi[d] + 1) * h) ** 2
                                         for d in range(3)))
                    far = math.sqrt(sum(max(abs(lo[d] * h - ctr[d]), abs((hi[d] + 1) * h - ctr[d])) ** 2
                                        for d in range(3)))
                    if near <= r + 2 * h and far >= r - 2 * h:
                        patches.append(ia.Patch(lo, hi, [v * h for v in lo], [(v + 1) * h for v in hi]))
                        break
    level = ia.Level([h] * 3, [0] * 3, [n - 1] * 3, [0.0] * 3, [1.0] * 3, [0] * 3, patches)
    return level, spheres


def _amr_inputs(c, seed):
    level, spheres = _amr_geometry(c)
    h = 1.0 / c["n"]
    g = _gen(seed)
    X = []
    left = c["points"]
    for i, (ctr, r) in enumerate(spheres):
        m = left if i == len(spheres) - 1 else c["points"] // len(spheres)
        left -= m
        X.append(torch.tensor(ctr, device=DEV, dtype=torch.float64) +
                 (r + h * (2 * _rand(g, m, 1) - 1)) * _directions(g, m, 3))
    X = _regrid_order(torch.cat(X), h, c["n"])
    F = _randn(g, c["points"], 3).to(_dtype(c["prec"]))
    gcw = [GHOST[c["kernel"]]] * 3
    flat, u = _pool(_shapes(level, gcw, ia.SIDE), _dtype(c["prec"]), g)
    # one velocity field over the level (a face two patches share has one value); the ghost values are still to fill
    k = (2 * math.pi * (1 + _rand(g, 3, 3) * 8)).cpu().tolist()
    for i, v in enumerate(u):
        P, a = level.patches[i // 3], i % 3
        x = [(torch.arange(P.ilower[d], P.iupper[d] + (2 if d == a else 1), device=DEV, dtype=torch.float64) +
              (0.0 if d == a else 0.5)) * h for d in range(3)]
        w = [torch.sin(k[a][d] * x[d] + d) for d in range(3)]
        v[tuple(slice(q, -q) for q in reversed(gcw))] = w[2][:, None, None] * w[1][:, None] * w[0]
    return level, gcw, X, F, u


def _box_level(n, cuts, periodic):
    """n cells per axis, the box cut into cuts^3 patches (unequal where it does
    not divide), spacing 1/n[0]."""
    h = 1.0 / n[0]
    e = [[(n[d] * i) // cuts for i in range(cuts + 1)] for d in range(3)]
    patches = []
    for k in range(cuts):
        for j in range(cuts):
            for i in range(cuts):
                lo = [e[0][i], e[1][j], e[2][k]]
                hi = [e[0][i + 1] - 1, e[1][j + 1] - 1, e[2][k + 1] - 1]
                patches.append(ia.Patch(lo, hi, [v * h for v in lo], [(v + 1) * h for v in hi]))
    return ia.Level([h] * 3, [0] * 3, [v - 1 for v in n], [0.0] * 3, [v * h for v in n],
                    list(n) if periodic else [0] * 3, patches)


def _ring_elements(c, seed):
    """Closed rings of nodes: springs between neighbours, beams along the ring,
    a target point at every c["every"]-th node (host arrays, node positions on
    the device)."""
    rng = np.random.default_rng(seed)
    n, rings = c["nodes"], min(c["rings"], c["nodes"] // 8)
    start = (np.arange(rings + 1) * n) // rings
    i = np.arange(n)
    ring = np.searchsorted(start, i, side="right") - 1
    s, m = start[ring], start[ring + 1] - start[ring]
    nxt, prv = s + (i - s + 1) % m, s + (i - s - 1) % m
    t = 2 * math.pi * (i - s) / m
    r = rng.uniform(0.05, 0.3, rings)[ring]
    X = np.stack([0.5 + r * np.cos(t), 0.5 + r * np.sin(t), rng.uniform(0.2, 0.8, rings)[ring]], axis=1)
    X = X + 1e-3 * rng.standard_normal(X.shape) * (r / m)[:, None]
    node = np.arange(0, n, c["every"])
    return {"X": X, "springs": (i, nxt, rng.uniform(1, 2, n), np.full(n, 1e-4)),
            "beams": (prv, i, nxt, rng.uniform(1e-3, 1e-2, n), np.zeros((n, 3))),
            "targets": (node, rng.uniform(1, 2, len(node)), rng.uniform(0, 1, len(node)),
                        X[node] + 1e-3 * rng.standard_normal((len(node), 3))),
            "U": rng.standard_normal((n, 3))}


def _fe_mesh(c, seed):
    """A box of Q1 elements with distorted nodes: positions and force density at
    the nodes, connectivity, shape function table, JxW."""
    nd, e = c["ndim"], c["edge"]
    g = _gen(seed)
    ax = [torch.arange(e + 1, device=DEV, dtype=torch.float64)] * nd
    grid = torch.meshgrid(*ax, indexing="ij")
    idx = torch.stack([v.reshape(-1) for v in reversed(grid)], dim=1)      # first axis fastest
    width = 0.4
    X = 0.3 + (width / e) * (idx + 0.15 * (2 * _rand(g, idx.shape[0], nd) - 1))
    corners = [(-1, -1), (1, -1), (1, 1), (-1, 1)]
    corners = corners if nd == 2 else [q + (z,) for z in (-1, 1) for q in corners]
    ei = torch.meshgrid(*([torch.arange(e, device=DEV)] * nd), indexing="ij")
    ei = [v.reshape(-1) for v in reversed(ei)]
    E = torch.stack([sum((ei[d] + (1 if q[d] > 0 else 0)) * (e + 1) ** d for d in range(nd)) for q in corners], dim=1)
    xi, w = fe.gauss_rule(nd, c["rule"])
    phi = torch.tensor(fe.q1_shape(nd, xi), device=DEV)
    dphi = torch.tensor(fe.q1_shape_grad(nd, xi), device=DEV)
    J = torch.stack([torch.stack([(X[E][:, :, d] @ dphi[j]) for j in range(nd)], dim=-1) for d in range(nd)], dim=-2)
    if nd == 2:
        det = J[..., 0, 0] * J[..., 1, 1] - J[..., 0, 1] * J[..., 1, 0]
    else:
        det = (J[..., 0, :] * torch.linalg.cross(J[..., 1, :], J[..., 2, :])).sum(-1)
    JxW = (det * torch.tensor(w, device=DEV)).contiguous()
    F = _randn(g, X.shape[0], nd)
    level = ia.Level.uniform_periodic(c["n"], nd)
    gcw = [GHOST[c["kernel"]]] * nd
    flat, u = _pool(_shapes(level, gcw, ia.SIDE), _dtype(c["prec"]), g)
    return level, gcw, X.contiguous(), F, E.to(torch.int32).contiguous(), phi.contiguous(), JxW, u


def _step_inputs(c, seed):
    k = c["shells"]
    rng = np.random.default_rng(7)   # the shells' sizes belong to the case
    w = np.exp(rng.uniform(0.0, math.log(100.0), k))
    counts = [max(8, int(v)) for v in c["points"] * w / w.sum()]
    structs = [("IB_4" if i < k // 2 else "BSPLINE_3", m) for i, m in enumerate(counts)]
    X = ibstep.ellipsoid_shells(k, counts, seed)
    n4 = sum(m for s, m in structs if s == "IB_4")
    h = 1.0 / c["n"]
    X = torch.cat([_regrid_order(X[:n4], h, c["n"]), _regrid_order(X[n4:], h, c["n"])]).contiguous()
    F = _randn(_gen(seed + 1), X.shape[0], 3).to(_dtype(c["prec"]))
    level = ia.Level.uniform_periodic(c["n"], 3)
    u_bg = ibstep.background_velocity(level, [3] * 3, _dtype(c["prec"]))
    return level, structs, X, F, u_bg, 0.05 * h ** 3, 0.5 * h


def _wall_inputs(c, seed):
    n = [c["nx"], c["ny"], c["nz"]]
    level = _box_level(n, c["cuts"], False)
    h = level.dx[0]
    side = c["centering"] == "side"
    gcw = [GHOST[c["kernel"]]] * 3
    g = _gen(seed)
    X = _rand(g, c["points"], 3)
    X[: c["points"] // 4, 2] *= 3.0 / n[2]                   # a quarter of the points near the bottom wall
    X = X * torch.tensor([v * h for v in n], device=DEV, dtype=torch.float64)
    key = _cells(X, h)
    X = X[torch.argsort((key[:, 2] * n[1] + key[:, 1]) * n[0] + key[:, 0], stable=True)].contiguous()
    fd = 3 if side else c["depth"]
    F = _randn(g, c["points"], fd).to(_dtype(c["prec"]))
    flat, u = _pool(_shapes(level, gcw, ia.SIDE if side else ia.CELL, c["depth"]), _dtype(c["prec"]), g)
    boxes, abg = [], []
    for p in range(len(level.patches)):
        for (codim, loc, lo, hi) in ia.physical_boundary_boxes(level, p, gcw[0]):
            boxes.append((p, codim, loc, lo, hi))
            # no slip at the walls, a moving lid at the upper z face
            abg.append([(1.0, 0.0, 1.0 if loc == 5 and a == 0 else 0.0) for a in range(fd)])
    return level, gcw, X, F, flat, u, boxes, np.array(abg).reshape(len(boxes), fd, 3)


# --------------------------------------------------------------------------- the state and the pass

def prepare(case, seed):
    c, k, dt_ = case, case["kind"], _dtype(case.get("prec", "fp64"))
    if k in ("ib", "amr"):
        level, gcw, X, F, u = _ib_inputs(c, seed) if k == "ib" else _amr_inputs(c, seed)
        plan = ia.LevelPlan(level, c["kernel"], ia.SIDE, _prec(c["prec"]), data_gcw=gcw, max_points=X.shape[0])
        flat, f = _pool(_shapes(level, gcw, ia.SIDE), dt_)
        plan.bind(0, f)
        plan.bind(1, u)
        plan.bin(X)
        if c["tune"]:
            plan.autotune(0, F, X, reps=2)
        return {"kind": k, "plan": plan, "f": flat, "X": X, "F": F, "U": torch.zeros_like(F),
                "Xn": torch.empty_like(X), "dt": 0.1 / c["n"]}
    if k == "walls":
        level, gcw, X, F, uflat, u, boxes, abg = _wall_inputs(c, seed)
        cen = ia.SIDE if c["centering"] == "side" else ia.CELL
        plan = ia.LevelPlan(level, c["kernel"], cen, _prec(c["prec"]), depth=c["depth"], data_gcw=gcw,
                            max_points=X.shape[0])
        flat, f = _pool(_shapes(level, gcw, cen, c["depth"]), dt_)
        plan.bind(0, f)
        plan.bind(1, u)
        plan.set_physical_boundary(boxes, abg)
        plan.bin(X)
        return {"kind": k, "plan": plan, "f": flat, "u": uflat, "X": X, "F": F, "U": torch.zeros_like(F)}
    if k == "step":
        level, structs, X, F, u_bg, alpha, dt = _step_inputs(c, seed)
        S = ibstep.StructureSet(level, structs, _prec(c["prec"]), alpha=alpha, u_bg=u_bg)
        U = torch.zeros_like(F)
        X0 = X.clone()
        S.step(X, F, U, dt)
        torch.cuda.synchronize()
        graph = S.capture(X, F, U, dt)
        X.copy_(X0)
        return {"kind": k, "set": S, "graph": graph, "X": X, "F": F, "U": U}
    if k == "regrid":
        level = _box_level([c["n"]] * 3, c["cuts"], True)
        g = _gen(seed)
        n = c["points"]
        X = torch.remainder(_points(g, n, 3, 1.0 / c["n"], "mixed") + 0.01 * _randn(g, n, 3), 1.0)
        plan = ia.LevelPlan(level, "IB_4", ia.SIDE, _prec(c["prec"]), max_points=n)
        F = _randn(g, n, 3).to(dt_)
        return {"kind": k, "plan": plan, "X": X.contiguous(), "F": F, "Xp": torch.empty_like(X),
                "Fp": torch.empty_like(F), "lag": torch.randperm(n, generator=g, device=DEV).to(torch.int32)}
    if k == "forces":
        e = _ring_elements(c, seed)
        X = torch.tensor(e["X"], device=DEV)
        f = structure.Forces(3, c["nodes"], springs=e["springs"], beams=e["beams"], targets=e["targets"])
        return {"kind": k, "forces": f, "X": X, "U": torch.tensor(e["U"], device=DEV).to(dt_),
                "F": torch.zeros(X.shape, dtype=dt_, device=DEV)}
    level, gcw, X, F, E, phi, JxW, u = _fe_mesh(c, seed)
    nq = JxW.numel()
    plan = ia.LevelPlan(level, c["kernel"], ia.SIDE, _prec(c["prec"]), data_gcw=gcw, max_points=nq)
    flat, f = _pool(_shapes(level, gcw, ia.SIDE), dt_)
    plan.bind(0, f)
    plan.bind(1, u)
    return {"kind": k, "plan": plan, "mesh": ia.FEMesh(E.cpu().numpy(), X.shape[0]), "f": flat, "X": X, "F": F,
            "E": E, "phi": phi, "JxW": JxW, "Uq": torch.zeros((nq, c["ndim"]), dtype=dt_, device=DEV),
            "rhs": torch.zeros_like(F)}


def run(state):
    s, k = state, state["kind"]
    if k == "ib":
        s["plan"].spread(0, s["F"], s["X"], mode=ia.OVERWRITE)
        s["plan"].fill_periodic_ghosts(1)
        s["plan"].interp(1, s["U"], None)   # at the spread's positions
        ia.forward_euler_step(s["Xn"], s["X"], s["U"], s["dt"])
        return {"f": s["f"], "U": s["U"], "X": s["Xn"]}
    if k == "amr":
        s["plan"].spread(0, s["F"], s["X"], mode=ia.OVERWRITE)
        s["plan"].fill_ghosts(1)
        s["plan"].interp(1, s["U"], s["X"])
        ia.forward_euler_step(s["Xn"], s["X"], s["U"], s["dt"])
        return {"f": s["f"], "U": s["U"], "X": s["Xn"]}
    if k == "walls":
        s["plan"].spread(0, s["F"], s["X"], mode=ia.OVERWRITE)
        s["plan"].accumulate_physical_boundary(0)
        s["plan"].fill_ghosts(1)
        s["plan"].fill_physical_boundary(1)
        s["plan"].interp(1, s["U"], s["X"])
        return {"f": s["f"], "u": s["u"], "U": s["U"]}
    if k == "step":
        s["graph"].replay()
        return {"X": s["X"], "U": s["U"], "f": list(s["set"].f)}
    if k == "regrid":
        order, patch_offsets, _ = s["plan"].redistribute(s["X"], s["lag"])
        ia.permute_rows(s["Xp"], s["X"], order)
        ia.permute_rows(s["Fp"], s["F"], order)
        s["plan"].bin(s["Xp"])
        return {"order": order, "offsets": patch_offsets, "X": s["Xp"], "F": s["Fp"]}
    if k == "forces":
        s["forces"].compute(s["F"], s["X"], s["U"])
        return {"F": s["F"]}
    Xq, Fq = ia.fe_quadrature_points(s["E"], s["phi"], s["JxW"], s["X"], s["F"], f_dtype=s["Uq"].dtype)
    s["plan"].bin(Xq, check=False)
    s["plan"].spread(0, Fq, Xq, mode=ia.OVERWRITE)
    s["plan"].fill_periodic_ghosts(1)
    s["plan"].interp(1, s["Uq"], None)
    s["mesh"].integrate_rhs(s["rhs"], s["Uq"], s["phi"], s["JxW"])
    return {"f": s["f"], "rhs": s["rhs"]}


# --------------------------------------------------------------------------- work

def _grid_values(level, gcw, centering, depth=1):
    return sum(int(np.prod(s)) for s in _shapes(level, gcw, centering, depth))


def _coupling_work(N, nd, fd, W, s, grid):
    """One spread into the whole arrays and one interpolation of N points: X and
    F read, every grid value written; X read, each stencil value read once (at
    most the whole arrays), U written."""
    touched = min(grid, N * fd * W ** nd)
    return {"bytes": N * (8 * nd + s * fd) + s * grid + N * (8 * nd + s * fd) + s * touched,
            "flops": 2 * N * fd * 3 * W ** nd}


def work(case):
    c, k = case, case["kind"]
    s = 8 if c.get("prec", "fp64") == "fp64" else 4
    if k == "forces":
        n, t = c["nodes"], c["nodes"] // c["every"]
        return {"bytes": n * (24 + 2 * 3 * s) + n * (8 + 16) + n * (12 + 8 + 24) + t * (4 + 16 + 24),
                "flops": n * (20 + 15 + 15) + 15 * t}
    if k == "regrid":
        n = c["points"]
        return {"bytes": n * (24 + 4 + 24 + 4) + n * (2 * 24 + 2 * 3 * s + 4) + n * (24 + 4 + 16), "flops": 0}
    if k == "step":
        level = ia.Level.uniform_periodic(c["n"], 3)
        grid = _grid_values(level, [3] * 3, ia.SIDE)
        n = c["points"]
        w = _coupling_work(n, 3, 3, 4, s, grid)
        # background and spread field read, velocity written; positions read and written; binned
        return {"bytes": w["bytes"] + 3 * s * grid + n * (48 + 3 * s) + n * (24 + 16), "flops": w["flops"]}
    W = WIDTH[c["kernel"]]
    if k == "fe":
        nd, e = c["ndim"], c["edge"]
        nq, nn, ne = (e * c["rule"]) ** nd, (e + 1) ** nd, e ** nd
        grid = _grid_values(ia.Level.uniform_periodic(c["n"], nd), [GHOST[c["kernel"]]] * nd, ia.SIDE)
        w = _coupling_work(nq, nd, nd, W, s, grid)
        return {"bytes": w["bytes"] + 3 * 8 * nd * nn + ne * 4 * 2 ** nd + 2 * 8 * nq + nq * (8 * nd + s * nd),
                "flops": w["flops"] + 3 * nq * nd * 2 ** nd * 2}
    if k == "walls":
        level = _box_level([c["nx"], c["ny"], c["nz"]], c["cuts"], False)
        cen = ia.SIDE if c["centering"] == "side" else ia.CELL
        grid = _grid_values(level, [GHOST[c["kernel"]]] * 3, cen, c["depth"])
        return _coupling_work(c["points"], 3, 3 if cen == ia.SIDE else c["depth"], W, s, grid)
    nd = 3 if k == "amr" else c["ndim"]
    level = _amr_geometry(c)[0] if k == "amr" else ia.Level.uniform_periodic(c["n"], nd)
    w = _coupling_work(c["points"], nd, nd, W, s, _grid_values(level, [GHOST[c["kernel"]]] * nd, ia.SIDE))
    return {"bytes": w["bytes"] + c["points"] * (16 * nd + s * nd), "flops": w["flops"]}


# --------------------------------------------------------------------------- 64-bit values

def _weights(kernel, t):
    """First index and weights ([n][W]) along one axis of points at t = (x -
    x_lower) / h, the value of index i lying at i + 1/2."""
    near = torch.floor(t + 0.5)
    if kernel == "PIECEWISE_LINEAR":
        lo = torch.floor(t - 0.5)
        b = t - 0.5 - lo
        return lo.long(), torch.stack([1 - b, b], 1)
    if kernel == "BSPLINE_3":
        c = torch.floor(t)
        d = t - c - 0.5
        return c.long() - 1, torch.stack([0.5 * (0.5 - d) ** 2, 0.75 - d * d, 0.5 * (0.5 + d) ** 2], 1)
    if kernel == "IB_4":
        lo = near - 2
        r = t - (lo + 1.5)
        q = torch.sqrt(1 + 4 * r * (1 - r))
        return lo.long(), torch.stack([3 - 2 * r - q, 3 - 2 * r + q, 1 + 2 * r + q, 1 + 2 * r - q], 1) / 8
    # the six-point kernel with three continuous derivatives (Bao, Kaye, Peskin
    # 2016): the weight furthest below solves 28 p^2 + beta p + gamma = 0, the
    # others follow from the even/odd sums and the moment conditions
    lo = near - 3
    r = 1 - t + lo + 2.5
    K = 59 / 60 - math.sqrt(29) / 20
    r2, r3 = r * r, r ** 3
    beta = 9 / 4 - 1.5 * (K + r2) + (22 / 3 - 7 * K) * r - 7 / 3 * r3
    gamma = 0.25 * (0.5 * (161 / 36 - 59 / 6 * K + 5 * K * K) * r2 + (-109 / 24 + 5 * K) / 3 * r2 * r2 +
                    5 / 18 * r3 * r3)
    p = (-beta + torch.sqrt(beta * beta - 112 * gamma)) / 56
    a, b, e = (3 * K - 1) / 12 * r + r3 / 12, (4 - 3 * K) / 6 * r - r3 / 6, (K + r2) / 8
    return lo.long(), torch.stack([p, -3 * p - 1 / 16 + e + a, 2 * p + 1 / 4 + b, 2 * p + 5 / 8 - 2 * e,
                                   -3 * p + 1 / 4 - b, p - 1 / 16 + e - a], 1)


def _axis_weights(kernel, X, h, axis):
    return [_weights(kernel, X[:, d] / h + (0.5 if d == axis else 0.0)) for d in range(X.shape[1])]


def _add_points(out, lo, kernel, X, V, h, axis, off):
    """Adds V * delta of the points (shifted by off cells) to the flat array of
    the box that starts at index lo, dropping what falls outside it."""
    nd = X.shape[1]
    n = list(reversed(out.shape))
    flat = out.view(-1)
    for part in torch.split(torch.arange(X.shape[0], device=DEV), 1 << 21):
        w = _axis_weights(kernel, X[part], h, axis)
        v = V[part] / h ** nd
        for e in np.ndindex(*([w[0][1].shape[1]] * nd)):
            at, val, ok, mul = 0, v, True, 1
            for d in range(nd):
                i = w[d][0] + (off[d] + e[d] - lo[d])
                ok = (i >= 0) & (i < n[d]) & ok
                at = at + i * mul
                mul *= n[d]
                val = val * w[d][1][:, e[d]]
            flat.index_add_(0, torch.where(ok, at, 0), torch.where(ok, val, 0.0))


def _spread_exact(level, gcw, kernel, X, F, total=None):
    """The ghosted side arrays of every patch: each patch takes the points (and
    periodic images) whose cell lies in its box grown by the ghost width."""
    nd, h = level.ndim, level.dx[0]
    cell = _cells(X, h)
    out = []
    for p, P in enumerate(level.patches):
        picked = []
        shifts = [(0, -1, 1) if s > 0 else (0,) for s in level.periodic_shift]
        for o in np.ndindex(*[len(s) for s in shifts]):
            off = [shifts[d][o[d]] * level.periodic_shift[d] for d in range(nd)]
            ok = torch.ones(X.shape[0], dtype=torch.bool, device=DEV)
            for d in range(nd):
                ok &= (cell[:, d] + off[d] >= P.ilower[d] - gcw[d]) & (cell[:, d] + off[d] <= P.iupper[d] + gcw[d])
            sel = torch.nonzero(ok).squeeze(1)
            if sel.numel():
                picked.append((off, sel))
        for a in range(nd):
            arr = torch.zeros(ia.array_shape(level, p, gcw, ia.SIDE, axis=a), dtype=torch.float64, device=DEV)
            for off, sel in picked:
                _add_points(arr, [P.ilower[d] - gcw[d] for d in range(nd)], kernel, X[sel], F[sel, a], h, a, off)
            out.append(arr)
    return out


def _interp_exact(level, gcw, kernel, X, u):
    nd, h = level.ndim, level.dx[0]
    cell = _cells(X, h)
    U = torch.zeros((X.shape[0], nd), dtype=torch.float64, device=DEV)
    for p, P in enumerate(level.patches):
        ok = torch.ones(X.shape[0], dtype=torch.bool, device=DEV)
        for d in range(nd):
            ok &= (cell[:, d] >= P.ilower[d]) & (cell[:, d] <= P.iupper[d])
        for part in torch.split(torch.nonzero(ok).squeeze(1), 1 << 21):
            for a in range(nd):
                arr = u[p * nd + a].to(torch.float64)
                n = list(reversed(arr.shape))
                flat, w, acc = arr.reshape(-1), _axis_weights(kernel, X[part], h, a), 0.0
                for e in np.ndindex(*([w[0][1].shape[1]] * nd)):
                    at, val, mul = 0, 1.0, 1
                    for d in range(nd):
                        at = at + (w[d][0] + (e[d] - P.ilower[d] + gcw[d])) * mul
                        mul *= n[d]
                        val = val * w[d][1][:, e[d]]
                    acc = acc + val * flat[at]
                U[part, a] = acc
    return U


def _wrap(arr, gcw, n):
    for d in range(arr.dim()):
        i = (torch.arange(arr.shape[d], device=DEV) - gcw) % n + gcw
        arr = arr.index_select(d, i)
    return arr


def _fill_level(level, gcw, u):
    """Ghost values that other patches of the level own, copied from them
    (through one array over the level, non-periodic)."""
    nd = level.ndim
    out = [v.clone() for v in u]
    for a in range(nd):
        n = [level.domain_upper[d] + 1 + 2 * gcw[d] + (1 if d == a else 0) for d in reversed(range(nd))]
        whole = torch.zeros(n, dtype=u[0].dtype, device=DEV)
        have = torch.zeros(n, dtype=torch.bool, device=DEV)

        def box(P, grow):
            return tuple(slice(P.ilower[d] + gcw[d] - grow * gcw[d],
                               P.iupper[d] + 1 + gcw[d] + grow * gcw[d] + (1 if d == a else 0))
                         for d in reversed(range(nd)))
        for p, P in enumerate(level.patches):
            core = tuple(slice(gcw[d], -gcw[d]) for d in reversed(range(nd)))
            whole[box(P, 0)] = u[p * nd + a][core]
            have[box(P, 0)] = True
        for p, P in enumerate(level.patches):
            w, b = whole[box(P, 1)], have[box(P, 1)].clone()
            b[tuple(slice(gcw[d], -gcw[d]) for d in reversed(range(nd)))] = False
            out[p * nd + a] = torch.where(b, w, out[p * nd + a])
    return out


def exact(case, seed):
    c, k = case, case["kind"]
    f64 = torch.float64
    if k == "ib":
        level, gcw, X, F, u = _ib_inputs(c, seed)
        f = _spread_exact(level, gcw, c["kernel"], X, F.to(f64))
        U = _interp_exact(level, gcw, c["kernel"], X, [_wrap(v, gcw[0], c["n"]) for v in u])
        return {"f": torch.cat([v.reshape(-1) for v in f]), "U": U, "X": X + 0.1 / c["n"] * U}
    if k == "amr":
        level, gcw, X, F, u = _amr_inputs(c, seed)
        f = _spread_exact(level, gcw, c["kernel"], X, F.to(f64))
        U = _interp_exact(level, gcw, c["kernel"], X, _fill_level(level, gcw, u))
        return {"f": torch.cat([v.reshape(-1) for v in f]), "U": U, "X": X + 0.1 / c["n"] * U}
    if k == "step":
        level, structs, X, F, u_bg, alpha, dt = _step_inputs(c, seed)
        n4 = sum(m for s, m in structs if s == "IB_4")
        f = None
        for kern, a, b in (("IB_4", 0, n4), ("BSPLINE_3", n4, X.shape[0])):
            g = _spread_exact(level, [3] * 3, kern, X[a:b], F[a:b].to(f64))
            f = g if f is None else [x + y for x, y in zip(f, g)]
        u = [_wrap(b.to(f64) + alpha * v, 3, c["n"]) for b, v in zip(u_bg, f)]
        U = torch.cat([_interp_exact(level, [3] * 3, kern, X[a:b], u)
                       for kern, a, b in (("IB_4", 0, n4), ("BSPLINE_3", n4, X.shape[0]))])
        return {"X": torch.remainder(X + dt * U, 1.0), "U": U, "f": f}
    if k == "forces":
        e = _ring_elements(c, seed)
        X, U = torch.tensor(e["X"], device=DEV), torch.tensor(e["U"], device=DEV).to(_dtype(c["prec"])).to(f64)
        t = lambda v: torch.tensor(v, device=DEV)  # noqa: E731
        m, s, kap, rest = (t(v) for v in e["springs"])
        D = X[s] - X[m]
        R = D.norm(dim=1)
        T = (kap * (R - rest) / R)[:, None] * D
        F = torch.zeros_like(X).index_add_(0, m, T).index_add_(0, s, -T)
        p, m, q, K, curv = (t(v) for v in e["beams"])
        B = K[:, None] * (X[q] + X[p] - 2 * X[m] - curv)
        F.index_add_(0, m, 2 * B).index_add_(0, q, -B).index_add_(0, p, -B)
        i, kap, eta, X0 = (t(v) for v in e["targets"])
        return {"F": F.index_add_(0, i, kap[:, None] * (X0 - X[i]) - eta[:, None] * U[i])}
    if k == "fe":
        level, gcw, X, F, E, phi, JxW, u = _fe_mesh(c, seed)
        nd, E = c["ndim"], E.long()
        Xq = torch.einsum("ekd,kq->eqd", X[E], phi).reshape(-1, nd)
        Fq = (torch.einsum("ekd,kq->eqd", F[E], phi) * JxW[:, :, None]).reshape(-1, nd)
        f = _spread_exact(level, gcw, c["kernel"], Xq, Fq)
        U = _interp_exact(level, gcw, c["kernel"], Xq, [_wrap(v, gcw[0], c["n"]) for v in u])
        r = torch.einsum("eqd,kq,eq->ekd", U.reshape(E.shape[0], -1, nd), phi, JxW)
        rhs = torch.zeros_like(X).index_add_(0, E.reshape(-1), r.reshape(-1, nd))
        return {"f": torch.cat([v.reshape(-1) for v in f]), "rhs": rhs}
    return None   # walls: no closed form beside the library's operators; regrid: copies only
