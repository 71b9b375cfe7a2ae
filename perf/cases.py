"""The work that users of meshoid_amd have it do, as timed cases.

A case is a dict of plain values.  ``listed()`` holds the fixed ones,
``draw(rng)`` gives further ones of the same ranges, ``prepare`` makes what a
program has in hand before the call, ``run`` is one pass through the public
entry points, ``work`` what a pass cannot do without, and ``exact`` the same
results in plain float64 torch.

Positions are uniform in the unit box, or clustered: Gaussian clumps with
log-uniform widths in [0.05, 5] and masses dN/dM ~ M^-2 in a 100-unit box plus
a 10% uniform background (six decades of density), stored clump by clump.
"""
from __future__ import annotations

import math

import torch

import meshoid_amd
from meshoid_amd import engine
from meshoid_amd.batch import SnapshotBatch

BOX = 100.0


def listed():
    return [
        # a notebook cell or a test: a few thousand particles in a periodic
        # box, density and one gradient; launches and latency count
        {"name": "periodic_4k", "kind": "meshoid", "n": 4096, "dim": 3, "dist": "uniform", "f64": True,
         "box": True, "k": 32, "order": 1, "comps": 1},
        # a small snapshot, the gradient of a velocity field
        {"name": "uniform_64k", "kind": "meshoid", "n": 65536, "dim": 3, "dist": "uniform", "f64": False,
         "box": False, "k": 32, "order": 1, "comps": 3},
        # a 2D simulation with its default neighbour number
        {"name": "plane_200k", "kind": "meshoid", "n": 200003, "dim": 2, "dist": "uniform", "f64": True,
         "box": False, "k": 20, "order": 1, "comps": 1},
        # second derivatives with many neighbours, as in the gradient notebook
        {"name": "hessian_1m_k100", "kind": "meshoid", "n": 1000000, "dim": 3, "dist": "uniform", "f64": True,
         "box": True, "k": 100, "order": 2, "comps": 1},
        # a clustered snapshot, density and the gradient of four fields
        {"name": "clustered_4m", "kind": "meshoid", "n": 1 << 22, "dim": 3, "dist": "clustered", "f64": False,
         "box": False, "k": 32, "order": 1, "comps": 4},
        # a program that steps a large snapshot through the device engine:
        # index build, neighbours, smoothing length, density, one gradient
        {"name": "engine_16m", "kind": "engine", "n": 1 << 24, "k": 32, "comps": 1},
        # many uneven snapshots, 32 fields each, through one graph launch
        {"name": "batch_16x32", "kind": "batch", "nsnap": 16, "n_lo": 1 << 14, "n_hi": 1 << 20, "K": 32},
        # neighbour rows, kernel weights and neighbour statistics of a snapshot
        {"name": "neighbours_250k", "kind": "stats", "n": 250000, "k": 32, "comps": 3},
        # two planes of sightlines cut through a snapshot whose lists exist
        {"name": "slices_512", "kind": "slices", "n": 1 << 21, "res": 512, "comps": 1},
        # a projected map and a volume of a snapshot with known radii
        {"name": "surface_1024", "kind": "surface", "n": 1 << 22, "res": 1024, "cons": False},
        {"name": "volume_128", "kind": "volume", "n": 1 << 22, "res": 128, "box": False},
        # emission and absorption along z, one band
        {"name": "radtransfer_128", "kind": "radtransfer", "n": 1 << 20, "res": 128, "bands": 1},
    ]


def _logn(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["meshoid", "meshoid", "meshoid", "engine", "batch", "stats", "slices", "surface", "volume",
                       "radtransfer"])
    if kind == "meshoid":
        order = rng.choice([1, 1, 2])
        dim = 3 if order == 2 else rng.choice([2, 3, 3])
        k = rng.choice([16, 20, 24]) if dim == 2 else rng.choice([20, 32, 32, 48, 64, 100])
        if order == 2:
            k = max(k, 48)  # nine coefficients per row
        uniform = dim == 2 or order == 2 or rng.random() < 0.5
        return {"kind": kind, "n": _logn(rng, 4000, 1 << (20 if k > 32 else 22)), "dim": dim,
                "dist": "uniform" if uniform else "clustered", "f64": rng.random() < 0.5 if uniform else False,
                "box": uniform and rng.random() < 0.5, "k": k, "order": order, "comps": rng.choice([1, 1, 3, 4])}
    if kind == "engine":
        return {"kind": kind, "n": _logn(rng, 1 << 18, 1 << 24), "k": rng.choice([24, 32, 32, 32]),
                "comps": rng.choice([1, 1, 2])}
    if kind == "batch":
        return {"kind": kind, "nsnap": rng.randint(4, 16), "n_lo": 1 << 14, "n_hi": _logn(rng, 1 << 16, 1 << 20),
                "K": rng.choice([8, 12, 32, 32])}
    if kind == "stats":
        return {"kind": kind, "n": _logn(rng, 5000, 300000), "k": rng.choice([20, 32, 32, 64]),
                "comps": rng.choice([1, 3])}
    if kind == "slices":
        return {"kind": kind, "n": _logn(rng, 1 << 15, 1 << 21), "res": _logn(rng, 64, 512), "comps": rng.choice([1, 3])}
    if kind == "surface":
        return {"kind": kind, "n": _logn(rng, 1 << 14, 1 << 22), "res": _logn(rng, 64, 1024), "cons": rng.random() < 0.5}
    if kind == "volume":
        return {"kind": kind, "n": _logn(rng, 1 << 14, 1 << 22), "res": _logn(rng, 32, 160), "box": rng.random() < 0.5}
    return {"kind": kind, "n": _logn(rng, 1 << 14, 1 << 20), "res": _logn(rng, 64, 160), "bands": rng.choice([1, 1, 3])}


# --------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _clustered(n, g, nclump=256, background=0.1):
    """((n, 3) float32 positions, clump centres, widths, particles per clump)."""
    c = _rand(g, nclump, 3) * BOX
    s = torch.exp(_rand(g, nclump) * math.log(100.0) + math.log(0.05))
    mass = 1.0 / (1.0 - _rand(g, nclump) * (1.0 - 1e-4))
    nbg = int(round(background * n))
    edge = torch.cumsum(mass, 0) / mass.sum()
    ids = torch.sort(torch.searchsorted(edge, _rand(g, n - nbg)).clamp(max=nclump - 1)).values
    pos = torch.empty(n, 3, device="cuda", dtype=torch.float32)
    pos[:nbg] = (_rand(g, nbg, 3) * BOX).float()
    pos[nbg:] = (c[ids] + s[ids, None] * torch.randn(n - nbg, 3, generator=g, device="cuda",
                                                     dtype=torch.float64)).float()
    return pos, c, s, torch.bincount(ids, minlength=nclump).double()


def _radii(pos, c, s, cnt, nbg):
    """Smoothing lengths of 32 neighbours in the clumps' own density."""
    out = torch.empty(pos.shape[0], device="cuda", dtype=torch.float64)
    amp = cnt / (s * math.sqrt(2 * math.pi)) ** 3
    for i in range(0, pos.shape[0], 1 << 18):
        p = pos[i:i + (1 << 18)].double()
        r2 = (p[:, None, 0] - c[:, 0]) ** 2 + (p[:, None, 1] - c[:, 1]) ** 2 + (p[:, None, 2] - c[:, 2]) ** 2
        dens = (amp * torch.exp(-0.5 * r2 / s**2)).sum(1) + nbg / BOX**3
        out[i:i + (1 << 18)] = (32.0 / (4 * math.pi / 3 * dens)) ** (1.0 / 3)
    return out


def _fields(pos, comps, wavelength, g):
    """Smooth float32/float64 fields sin(k x + p) sin(k y + p) (sin(k z + p))."""
    ph = _rand(g, comps) * 0.5
    x = pos.double() * (2 * math.pi / wavelength)
    f = torch.ones(pos.shape[0], comps, device="cuda", dtype=torch.float64)
    for a in range(pos.shape[1]):
        f *= torch.sin(x[:, a, None] + ph)
    f = f.to(pos.dtype).contiguous()
    return f[:, 0].contiguous() if comps == 1 else f


def _points(case, g):
    """Positions, box length and the wavelength of the fields of a point set."""
    if case.get("dist", "clustered") == "uniform":
        pos = _rand(g, case["n"], case["dim"])
        return (pos if case["f64"] else pos.float()).contiguous(), (1.0 if case["box"] else None), 1.0
    return _clustered(case["n"], g)[0], None, 10.0


def _sizes(case):
    """Particles per snapshot, spread over the logarithm of the range."""
    m = case["nsnap"]
    at = [((7 * s + 3) % m + 0.5) / m if m % 7 else (s + 0.5) / m for s in range(m)]
    return [int(round(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** t)) for t in at]


def _snapshots(case, g):
    sizes = _sizes(case)
    pos, fields = [], []
    for s, n in enumerate(sizes):
        p = _clustered(n, g, nclump=8 + (s * 37) % 121)[0]
        q = p.double() / BOX
        a = torch.randn(3, case["K"], generator=g, device="cuda", dtype=torch.float64)
        f = torch.randn(n, case["K"], generator=g, device="cuda", dtype=torch.float64) + q @ a + (q * q) @ a.flip(0)
        pos.append(p)
        fields.append(f.float().contiguous())
    return sizes, [32 if s % 2 == 0 else 64 for s in range(len(sizes))], pos, fields


def _planes(case, g):
    """Two planes z = const of res x res points through the clumps' box."""
    ax = torch.linspace(20.0, 80.0, case["res"], device="cuda", dtype=torch.float64)
    x, y = torch.meshgrid(ax, ax, indexing="ij")
    zs = 30.0 + 40.0 * _rand(g, 2).sort().values
    return [torch.stack((x.reshape(-1), y.reshape(-1), torch.full_like(x, float(z)).reshape(-1)), 1).contiguous()
            for z in zs]


def _deposit(case, g):
    pos, c, s, cnt = _clustered(case["n"], g)
    h = _radii(pos, c, s, cnt, int(round(0.1 * case["n"])))
    m = (0.5 + _rand(g, case["n"])) / case["n"]
    return pos, h, m


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "meshoid":
        pos, box, lam = _points(case, g)
        return {"case": case, "pos": pos, "box": box, "f": _fields(pos, case["comps"], lam, g)}
    if kind == "engine":
        pos = _clustered(case["n"], g)[0]
        f = _fields(pos, case["comps"], 10.0, g).reshape(case["n"], -1)
        # a stepping program keeps its index, list and output buffers
        return {"case": case, "pos": pos, "f": f, "index": engine.SpatialIndex(), "nlist": engine.NeighborList()}
    if kind == "batch":
        sizes, ks, pos, fields = _snapshots(case, g)
        return {"case": case, "pos": pos, "fields": fields, "batch": SnapshotBatch(sizes, ks, case["K"])}
    if kind == "stats":
        pos = _clustered(case["n"], g)[0]
        f = _fields(pos, case["comps"], 10.0, g).reshape(case["n"], -1).contiguous()
        ix = engine.SpatialIndex().build(pos)
        nl = engine.knn_hsml(ix, case["k"], keep_dist=False)["nlist"]
        return {"case": case, "pos": pos, "f": f, "f0": f[:, 0].contiguous(), "index": ix, "nlist": nl}
    if kind == "slices":
        pos = _clustered(case["n"], g)[0]
        f = _fields(pos, case["comps"], 10.0, g)
        return {"case": case, "f": f, "planes": _planes(case, g), "meshoid": meshoid_amd.Meshoid(pos)}
    if kind in ("surface", "volume"):
        pos, h, m = _deposit(case, g)
        return {"case": case, "pos": pos, "h": h, "m": m}
    pos, h, m = _deposit(case, g)
    x = pos.double()
    kap = 3.0e4 * (0.5 + _rand(g, case["n"], case["bands"]))
    j = 0.5 + _rand(g, case["n"], case["bands"])
    return {"case": case, "x": x, "h": h, "m": m, "j": j, "kappa": kap}


# ------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "meshoid":
        M = meshoid_amd.Meshoid(state["pos"], des_ngb=case["k"], boxsize=state["box"])
        d = M.D(state["f"]) if case["order"] == 1 else M.D2(state["f"])
        a = M.device_arrays()
        return {"h": a["kernel_radius"], "density": a["density"], "vol": a["vol"], "d": d}
    if kind == "engine":
        state["index"].build(state["pos"])
        out = engine.knn_hsml(state["index"], case["k"], keep_dist=False, nlist=state["nlist"])
        d, _, _ = engine.apply_D(state["nlist"], state["f"])
        return {"h": out["h"], "rho": out["rho"], "vol": out["vol"], "d": d}
    if kind == "batch":
        o = state["batch"].run(state["pos"], state["fields"])
        return {"h": o["h"], "rho": o["rho"], "grad": o["grad"]}
    if kind == "stats":
        nl = state["nlist"]
        ngb, dist = nl.export(f64=True)
        return {"ngb": ngb, "dist": dist, "weights": engine.kernel_weights_dev(dist, nl.h64()),
                "average": engine.kernel_average(nl, state["f0"]), "sigma": engine.kernel_variance(nl, state["f"])}
    if kind == "slices":
        return [state["meshoid"].Reconstruct(state["f"], p) for p in state["planes"]]
    if kind == "surface":
        return meshoid_amd.GridSurfaceDensity(state["m"], state["pos"], state["h"].clamp(min=2 * BOX / case["res"]),
                                              (BOX / 2, BOX / 2, BOX / 2), BOX, case["res"],
                                              conservative=case["cons"])
    if kind == "volume":
        return meshoid_amd.GridDensity(state["m"], state["pos"], state["h"].clamp(min=BOX / (case["res"] - 1)),
                                       (BOX / 2, BOX / 2, BOX / 2), BOX, case["res"],
                                       box_size=BOX if case["box"] else -1.0)
    return meshoid_amd.radtransfer(state["j"], state["m"], state["kappa"], state["x"], state["h"], case["res"], BOX,
                                   center=(BOX / 2, BOX / 2, BOX / 2))


def _pairs(n, k, dim, order, comps):
    """Flops of the k neighbour terms of n rows: distance, two kernel sums of
    the smoothing length, moments and right-hand sides of the fit."""
    nd = dim if order == 1 else 9
    return n * k * (3 * dim + 40 + 2 * nd * (nd + 1) / 2 + 2 * nd * comps)


def work(case):
    """Bytes: inputs read once and outputs written once; flops: the terms of
    the k neighbours of each row, or the kernel at each cell of a footprint."""
    kind = case["kind"]
    if kind == "meshoid":
        n, dim, K = case["n"], case["dim"], case["comps"]
        e = 8 if case["f64"] else 4
        nd = dim if case["order"] == 1 else 6
        return {"bytes": n * (e * dim + e * K + 24 + 4 * nd * K), "flops": _pairs(n, case["k"], dim, case["order"], K)}
    if kind == "engine":
        n, K = case["n"], case["comps"]
        return {"bytes": n * (12 + 4 * K + 12 + 12 * K), "flops": _pairs(n, case["k"], 3, 1, K)}
    if kind == "batch":
        n = sum(_sizes(case))
        return {"bytes": n * (12 + 8 + 16 * case["K"]), "flops": _pairs(n, 48, 3, 1, case["K"])}
    if kind == "stats":
        n, k, K = case["n"], case["k"], case["comps"]
        return {"bytes": n * (12 + 4 * k + 20 * k + 8 + 8 * K), "flops": n * k * (9 + 15 + 15 + 4 * K)}
    if kind == "slices":
        npt = 2 * case["res"] ** 2
        return {"bytes": npt * (24 + 12 + 4 * case["comps"] + 4 * case["comps"]),
                "flops": _pairs(npt, 32, 3, 1, case["comps"])}
    if kind == "surface":
        # a clump particle's footprint is the smallest, 4 x 4 cells
        return {"bytes": case["n"] * 24 + 8 * case["res"] ** 2, "flops": case["n"] * 16 * 15}
    if kind == "volume":
        return {"bytes": case["n"] * 28 + 8 * case["res"] ** 3, "flops": case["n"] * 8 * 2 * 15}
    return {"bytes": case["n"] * (24 + 16 + 16 * case["bands"]) + 8 * case["res"] ** 2 * case["bands"],
            "flops": case["n"] * 4 * (15 + 30 * case["bands"])}


# -------------------------------------------------------- the same in 64 bits
def _image(d, box):
    """Offsets to the nearest periodic image."""
    if box is None:
        return d
    a = d.abs()
    return torch.where(a > box / 2, -torch.copysign(box - a, d), d)


def _knn_brute(pos, k, box):
    """(distances, indices) of the k nearest, ascending, by all pairs."""
    n = pos.shape[0]
    step = max(1, int(2.5e8) // n)
    dist = torch.empty(n, k, device="cuda", dtype=torch.float64)
    ngb = torch.empty(n, k, device="cuda", dtype=torch.int64)
    for i in range(0, n, step):
        d2 = 0.0
        for a in range(pos.shape[1]):
            d2 = d2 + _image(pos[None, :, a] - pos[i:i + step, None, a], box) ** 2
        v, j = torch.topk(d2, k, largest=False, sorted=True)
        dist[i:i + step], ngb[i:i + step] = v.sqrt(), j
    return dist, ngb


def _knn_cells(pos, k, box):
    """The same for uniform points in the unit cube: the 27 cells around each
    point, cells wider than the farthest k-th neighbour (checked)."""
    n = pos.shape[0]
    m = int((4.18879 * n / (k * 1.9)) ** (1.0 / 3))
    cell = (pos * m).long().clamp(max=m - 1)
    cid = (cell[:, 0] * m + cell[:, 1]) * m + cell[:, 2]
    order = torch.argsort(cid)
    cnt = torch.bincount(cid, minlength=m**3)
    first = torch.cumsum(cnt, 0) - cnt
    cap = int(cnt.max())
    dist = torch.empty(n, k, device="cuda", dtype=torch.float64)
    ngb = torch.empty(n, k, device="cuda", dtype=torch.int64)
    off = torch.stack(torch.meshgrid(*[torch.arange(-1, 2, device="cuda")] * 3, indexing="ij"), -1).reshape(-1, 3)
    lane = torch.arange(cap, device="cuda")
    step = max(1, int(1.2e8) // (27 * cap))
    for i in range(0, n, step):
        c = cell[i:i + step, None, :] + off
        ok = ((c >= 0) & (c < m)).all(-1) if box is None else torch.ones(c.shape[:2], device="cuda", dtype=torch.bool)
        c = c % m
        q = (c[..., 0] * m + c[..., 1]) * m + c[..., 2]
        valid = ((lane < cnt[q][..., None]) & ok[..., None]).reshape(c.shape[0], -1)
        cand = order[(first[q][..., None] + lane).clamp(max=n - 1)].reshape(c.shape[0], -1)
        d2 = 0.0
        for a in range(3):
            d2 = d2 + _image(pos[cand, a] - pos[i:i + step, None, a], box) ** 2
        v, j = torch.topk(torch.where(valid, d2, torch.inf), k, largest=False, sorted=True)
        dist[i:i + step], ngb[i:i + step] = v.sqrt(), torch.gather(cand, 1, j)
    if box is not None and float(dist.max()) > 1.0 / m:
        return None
    if box is None:
        # open faces: outer points need the cell width only inside the cube
        if float(dist.max()) > 1.0 / m:
            far = dist[:, -1] > 1.0 / m
            if int(far.sum()) > 20000:
                return None
            for i in torch.nonzero(far).reshape(-1).split(max(1, int(2.5e8) // n)):
                d2 = 0.0
                for a in range(3):
                    d2 = d2 + (pos[None, :, a] - pos[i, None, a]) ** 2
                v, j = torch.topk(d2, k, largest=False, sorted=True)
                dist[i], ngb[i] = v.sqrt(), j
    return dist, ngb


def _neighbours(pos, k, box, uniform):
    n, dim = pos.shape
    if n * n <= 1.6e11:
        return _knn_brute(pos, k, box)
    if uniform and dim == 3 and n * k <= 1.2e8:
        return _knn_cells(pos, k, box)
    return None


def _spline(q):
    a = 1.0 - q
    w = torch.where(q <= 0.5, 1.0 - 6.0 * q * q * a, 2.0 * a * a * a)
    return torch.where(q <= 1.0, w, torch.zeros_like(w))


def _hsml(dist, dim):
    """Root of norm sum_j W(r_j / h) = k by bisection."""
    k = dist.shape[1]
    norm = {2: 40.0 / 7, 3: 32.0 / 3}[dim]
    lo, hi = dist[:, 1].clone(), {2: 1.7984058958344455, 3: 1.5638742363463305}[dim] * dist[:, -1]
    for _ in range(56):
        h = 0.5 * (lo + hi)
        big = norm * _spline(dist / h[:, None]).sum(1) > k
        hi, lo = torch.where(big, h, hi), torch.where(big, lo, h)
    return 0.5 * (lo + hi)


def _fit(pos, ngb, h, f, box, order, rows):
    """Least-squares derivatives of f (n, K) at the given rows."""
    d = _image(pos[ngb[rows]] - pos[rows, None, :], box)
    w = _spline(d.norm(dim=2) / h[rows, None])
    if order == 2:
        x, y, z = d.unbind(2)
        d = torch.stack((x, y, z, x * x / 2, y * y / 2, z * z / 2, x * y, y * z, z * x), 2)
    # columns brought to one scale before the solve
    s = (w[..., None] * d * d).sum(1).sqrt()
    a = d / s[:, None, :]
    wa = (w[..., None] * a).transpose(1, 2).contiguous()
    E = torch.matmul(wa, a)
    b = torch.matmul(wa, (f[ngb[rows]] - f[rows, None, :]).contiguous())
    g = torch.linalg.solve(E, b) / s[:, :, None]
    return g.transpose(1, 2)  # (rows, K, columns)


def _derivatives(pos, ngb, h, f, box, order):
    n, dim = pos.shape
    out = torch.empty(n, f.shape[1], dim if order == 1 else 6, device="cuda", dtype=torch.float64)
    step = max(1, int(4e7) // (ngb.shape[1] * max(f.shape[1], 9)))
    for i in range(0, n, step):
        rows = torch.arange(i, min(n, i + step), device="cuda")
        g = _fit(pos, ngb, h, f, box, order, rows)
        out[rows] = g if order == 1 else g[:, :, 3:]
    return out


def _nearest_rows(x, pos, k):
    """_knn_brute of the points x."""
    step = max(1, int(2.5e8) // pos.shape[0])
    out = []
    for i in range(0, x.shape[0], step):
        d2 = 0.0
        for a in range(pos.shape[1]):
            d2 = d2 + (pos[None, :, a] - x[i:i + step, None, a]) ** 2
        v, j = torch.topk(d2, k, largest=False, sorted=True)
        out.append((v.sqrt(), j))
    return torch.cat([v for v, _ in out]), torch.cat([j for _, j in out])


def _slices_exact(case, pos, f, planes):
    if 4 * case["res"] ** 2 * pos.shape[0] > 8e10:
        return None
    out = []
    for x in planes:
        near = _nearest_rows(x, pos, 1)[1][:, 0]
        rows, inv = torch.unique(near, return_inverse=True)
        dist, ngb_r = _nearest_rows(pos[rows], pos, 32)
        ngb, h = torch.zeros(pos.shape[0], 32, device="cuda", dtype=torch.int64), torch.zeros_like(pos[:, 0])
        ngb[rows], h[rows] = ngb_r, _hsml(dist, 3)
        g = torch.cat([_fit(pos, ngb, h, f, None, 1, r) for r in rows.split(1 << 16)])[inv]
        v = f[near] + ((x - pos[near])[:, None, :] * g).sum(2)
        out.append(v[:, 0] if case["comps"] == 1 else v)
    return out


def _cells_of(x, h, dx, res, clip):
    lo, hi = ((x - h) / dx + 1.0), ((x + h) / dx)
    if clip:
        return lo.clamp(0, res).trunc().long(), torch.where(hi > -1.0, hi.clamp(max=res - 1.0).trunc(), -1.0).long()
    return lo.trunc().long(), hi.trunc().long()


def _spread(rel, h, spans, first, visit):
    """visit(particles, cells) over every footprint cell, offset by offset;
    particles whose span covers the offset only."""
    top = [int(s.max()) for s in spans]
    sel0 = torch.nonzero((spans[0] > 0) & (spans[1] > 0) & (spans[-1] > 0)).reshape(-1)
    for i in range(top[0]):
        si = sel0[spans[0][sel0] > i]
        for j in range(top[1]):
            sj = si[spans[1][si] > j]
            if sj.numel() == 0:
                break
            if len(spans) == 2:
                visit(sj, (first[0][sj] + i, first[1][sj] + j))
                continue
            for k in range(top[2]):
                sk = sj[spans[2][sj] > k]
                if sk.numel() == 0:
                    break
                visit(sk, (first[0][sk] + i, first[1][sk] + j, first[2][sk] + k))


def _map_exact(case, state):
    res, ndim = case["res"], 2 if case["kind"] == "surface" else 3
    wrap = case["kind"] == "volume" and case["box"]
    cons = case["kind"] == "volume" or case["cons"]
    dx = BOX / (res - 1)
    x = state["pos"].double()[:, :ndim] - (BOX / 2 - 0.5 * BOX) - (0.5 * dx if ndim == 3 else 0.0)
    h = state["h"].clamp(min=2 * BOX / res if ndim == 2 else dx)
    if cons and ndim == 2:
        h = h.clamp(min=dx)
    fl = [_cells_of(x[:, a], h, dx, res, not wrap) for a in range(ndim)]
    first, spans = [a for a, _ in fl], [b - a + 1 for a, b in fl]
    if float(torch.stack([s.clamp(min=0).double() for s in spans]).prod(0).sum()) > 3e9:
        return None
    norm = 40.0 / (7 * math.pi) if ndim == 2 else 8.0 / math.pi
    tot = torch.zeros_like(h)
    # 64 copies of the grid, one per residue of the particle number: a clump's
    # particles land on the same few cells
    grid = torch.zeros(64 * res**ndim, device="cuda", dtype=torch.float64)

    def weight(p, cells):
        r2 = 0.0
        for a in range(ndim):
            r2 = r2 + (x[p, a] - cells[a].double() * dx) ** 2
        return norm * _spline(r2.sqrt() / h[p])

    def total(p, cells):
        tot[p] += weight(p, cells)

    def add(p, cells):
        v = weight(p, cells) * state["m"][p]
        v = torch.where(tot[p] > 0, v / tot[p], 0.0) if cons else v / h[p] ** 2
        at = cells[0] % res
        for c in cells[1:]:
            at = at * res + c % res
        grid.index_add_(0, at + (p % 64) * res**ndim, v)

    if cons:
        _spread(x, h, spans, first, total)
    _spread(x, h, spans, first, add)
    grid = grid.reshape(64, -1).sum(0)
    return (grid / dx**ndim if cons else grid).reshape((res,) * ndim)


def _light_exact(case, state):
    """I = sum over a pixel's particles of S (1 - exp(-tau)) exp(-depth of the
    nearer ones); the depths from integer prefix sums, exact to 2^-60."""
    res, nf = case["res"], case["bands"]
    dx = BOX / (res - 1)
    xy = state["x"][:, :2] - (BOX / 2 - 0.5 * BOX)
    h = state["h"].clamp(min=dx)
    order = torch.argsort(state["x"][:, 2], descending=True, stable=True)
    rank = torch.empty_like(order)
    rank[order] = torch.arange(order.numel(), device="cuda")
    fl = [_cells_of(xy[:, a], h, dx, res, True) for a in range(2)]
    first, spans = [a for a, _ in fl], [b - a + 1 for a, b in fl]
    if float(torch.stack([s.clamp(min=0).double() for s in spans]).prod(0).sum()) > 2e8:
        return None
    parts, keys, kern = [], [], []

    def visit(p, cells):
        r2 = (xy[p, 0] - cells[0].double() * dx) ** 2 + (xy[p, 1] - cells[1].double() * dx) ** 2
        ok = r2 <= h[p] ** 2
        p = p[ok]
        parts.append(p)
        keys.append(((cells[0] * res + cells[1])[ok] << 32) | rank[p])
        kern.append(40.0 / (7 * math.pi) * _spline(r2[ok].sqrt() / h[p]) * state["m"][p] / h[p] ** 2)

    _spread(xy, h, spans, first, visit)
    key, at = torch.sort(torch.cat(keys))
    p, w, pix = torch.cat(parts)[at], torch.cat(kern)[at], key >> 32
    last = torch.searchsorted(pix, torch.arange(res * res, device="cuda"), right=True) - 1
    out = torch.empty(res * res, nf, device="cuda", dtype=torch.float64)
    copy = (torch.arange(pix.numel(), device="cuda") % 64) * (res * res) + pix
    for b in range(nf):
        tau = state["kappa"][p, b] * w
        hi = torch.floor(tau * 2.0**30)
        lo = torch.floor((tau * 2.0**30 - hi) * 2.0**30).long()
        chi, clo = torch.cumsum(hi.long(), 0), torch.cumsum(lo, 0)
        e = last[pix]
        near = (chi[e] - chi).double() * 2.0**-30 + (clo[e] - clo).double() * 2.0**-60
        src = state["j"][p, b] / (4 * math.pi * state["kappa"][p, b] + 1e-100)
        light = torch.zeros(64 * res * res, device="cuda", dtype=torch.float64)
        light.index_add_(0, copy, -torch.expm1(-tau) * src * torch.exp(-near))
        out[:, b] = light.reshape(64, -1).sum(0)
    return out.reshape(res, res, nf)


def exact(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind in ("meshoid", "engine"):
        pos, box, lam = _points(case, g)
        f = _fields(pos, case["comps"], lam, g).double().reshape(case["n"], -1)
        p64 = pos.double()
        found = _neighbours(p64, case["k"], box, case.get("dist") == "uniform")
        if found is None:
            return None
        dist, ngb = found
        dim = p64.shape[1]
        h = _hsml(dist, dim)
        vol = (math.pi if dim == 2 else 4 * math.pi / 3) * h**dim / case["k"]
        d = _derivatives(p64, ngb, h, f, box, case.get("order", 1))
        if kind == "engine":
            return {"h": h, "rho": 1.0 / vol, "vol": vol, "d": d}
        return {"h": h, "density": 1.0 / vol, "vol": vol, "d": d[:, 0] if case["comps"] == 1 else d}
    if kind == "batch":
        sizes, ks, pos, fields = _snapshots(case, g)
        out = {"h": [], "rho": [], "grad": []}
        for n, k, p, f in zip(sizes, ks, pos, fields):
            if n > 100000:
                for v in out.values():
                    v.append(None)
                continue
            p64 = p.double()
            dist, ngb = _knn_brute(p64, k, None)
            h = _hsml(dist, 3)
            out["h"].append(h)
            out["rho"].append(k / (4 * math.pi / 3 * h**3))
            out["grad"].append(_derivatives(p64, ngb, h, f.double(), None, 1))
        return out
    if kind == "stats":
        pos = _clustered(case["n"], g)[0]
        f = _fields(pos, case["comps"], 10.0, g).double().reshape(case["n"], -1)
        found = _neighbours(pos.double(), case["k"], None, False)
        if found is None:
            return None
        dist, ngb = found
        w = _spline(dist / _hsml(dist, 3)[:, None])
        w = w / w.sum(1, keepdim=True)
        fn = f[ngb]
        return {"ngb": None, "dist": dist, "weights": w, "average": (w * fn[..., 0]).sum(1),
                "sigma": fn.std(dim=1, correction=0)}
    if kind == "slices":
        pos = _clustered(case["n"], g)[0].double()
        f = _fields(pos.float(), case["comps"], 10.0, g).double().reshape(case["n"], -1)
        return _slices_exact(case, pos, f, _planes(case, g))
    if kind in ("surface", "volume"):
        pos, h, m = _deposit(case, g)
        return _map_exact(case, {"pos": pos, "h": h, "m": m})
    st = prepare(case, seed)
    return _light_exact(case, st)
