"""The workloads of fasttree_amd whose speed is followed.

Each case is one call sequence that a user's program makes through the public
entry points (`fasttree_amd`, `fasttree_amd.batch`, `fasttree_amd.learned` and
the C ABI they bind), with its inputs already on the GPU.  `listed()` names the
workloads, `draw()` gives more of the same ranges, `prepare()` makes a case's
inputs and the handles that a program keeps, `run()` is one pass, `work()` what
a pass cannot do without, and `exact()` the outputs in 64 bits where plain
tensor code can give them.

Snapshots are those of the package's own generator (`fasttree_amd.synth`): 70 %
of the particles in NFW halos of about 3,500 particles each, 30 % uniform
background, in a periodic box of side 100; here they are drawn on the GPU.
"""
import math

import numpy as np
import torch

import fasttree_amd as ft
from fasttree_amd.batch import Batch, plan_requests
from fasttree_amd.learned import MLP, NF, NPARAM, init_params

BOX = 100.0
BITS = 21
COORDS = {"f32": ft.COORD_F32, "f64": ft.COORD_F64, "i32": ft.COORD_U32, "i64": ft.COORD_U64}
SIZES = {"f32": 4, "f64": 8, "i32": 4, "i64": 8}
TORCH = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32, "i64": torch.int64}
CURVES = {"morton": ft.SFC_MORTON, "hilbert": ft.SFC_PEANO_HILBERT}


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest whole step: a simulation or a test program that rebuilds
        # a small tree and asks for every particle's neighbours, double
        # coordinates, 30-bit Morton keys.
        {"name": "step_f64_100k_k16", "kind": "step", "coord": "f64", "curve": "morton",
         "bits": 10, "periodic": False, "points": "uniform", "n": 100_000, "k": 16},
        # The same step of an ordinary size, with single-precision positions as
        # snapshots store them and an odd particle count.
        {"name": "step_f32_1m_k8", "kind": "step", "coord": "f32", "curve": "hilbert",
         "bits": BITS, "periodic": False, "points": "clustered", "n": 1_000_003, "k": 8},
        # The production build: 10M clustered fixed-point particles.
        {"name": "build_i64_10m", "kind": "build", "coord": "i64", "curve": "hilbert",
         "bits": BITS, "periodic": True, "points": "clustered", "n": 10_000_000, "ids": False},
        # The headline query: every particle's 32 nearest neighbours.
        {"name": "self_i64_10m_k32", "kind": "self", "coord": "i64", "curve": "hilbert",
         "bits": BITS, "periodic": True, "points": "clustered", "n": 10_000_000, "k": 32},
        # SPH with individual time steps: the neighbours of the active fifth of
        # a double-precision snapshot, k = 64.
        {"name": "subset_f64_20m_k64", "kind": "subset", "coord": "f64", "curve": "hilbert",
         "bits": BITS, "periodic": True, "points": "clustered", "n": 20_000_000,
         "queries": 4_000_000, "k": 64},
        # A handful of points looked up in a large tree (probes, sink particles,
        # an interactive query): latency counts.
        {"name": "knn_i64_1000q_k32", "kind": "knn", "coord": "i64", "curve": "hilbert",
         "bits": BITS, "periodic": True, "points": "clustered", "n": 10_000_000,
         "queries": 1000, "k": 32},
        # A set of tracer points against a 32-bit tree in an open box, small k.
        {"name": "knn_i32_500k_k8", "kind": "knn", "coord": "i32", "curve": "morton",
         "bits": BITS, "periodic": False, "points": "clustered", "n": 2_000_000,
         "queries": 500_000, "k": 8},
        # Density estimation at external points with many neighbours.
        {"name": "knn_i64_1m_k128", "kind": "knn", "coord": "i64", "curve": "hilbert",
         "bits": BITS, "periodic": True, "points": "clustered", "n": 10_000_000,
         "queries": 1_000_000, "k": 128},
        # SPH neighbour lists: every particle within 1.2 times its own 32nd
        # neighbour's distance, as counts and then a CSR list.
        {"name": "csr_f64_5m", "kind": "csr", "coord": "f64", "curve": "hilbert",
         "bits": BITS, "periodic": True, "points": "clustered", "n": 5_000_000},
        # Friends-of-friends linking: the particles within 0.2 mean separations
        # of each of a set of points, at most 64 kept per point.
        {"name": "range_i64_200k", "kind": "range", "coord": "i64", "curve": "hilbert",
         "bits": BITS, "periodic": True, "points": "clustered", "n": 3_000_000,
         "queries": 200_000, "cap": 64},
        # Many small and middle-sized trees rebuilt and queried as one captured
        # step, requests of mixed k (serving, zoom regions, several snapshots).
        {"name": "batch_i32_24trees", "kind": "batch", "coord": "i32", "curve": "morton",
         "bits": BITS, "periodic": False, "points": "clustered", "trees": 24, "n_min": 10_000,
         "n_max": 400_000, "queries": 300_000},
        # Training of the learned radius: forward and backward over one batch.
        {"name": "grad_64k", "kind": "grad", "rows": 65_536},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "build", "self", "subset", "knn", "knn", "csr", "range", "batch",
                       "grad"])
    if kind == "grad":
        return {"kind": kind, "rows": _log(rng, 4096, 262_144)}
    if kind == "batch":
        return {"kind": kind, "coord": rng.choice(["i32", "i64"]), "curve": "morton", "bits": BITS,
                "periodic": False, "points": "clustered", "trees": rng.randint(4, 32),
                "n_min": 10_000, "n_max": _log(rng, 50_000, 400_000),
                "queries": _log(rng, 20_000, 300_000)}
    coord = rng.choice(["f32", "f64", "i32", "i64"])
    # single precision has no periodic snapshots here; the others have both
    periodic = coord != "f32" and rng.random() < 0.6
    c = {"kind": kind, "coord": coord, "curve": rng.choice(["morton", "hilbert"]), "bits": BITS,
         "periodic": periodic, "points": rng.choice(["clustered", "clustered", "uniform"])}
    if kind == "build":
        return dict(c, n=_log(rng, 20_000, 10_000_000), ids=rng.random() < 0.3)
    if kind in ("step", "self"):
        return dict(c, n=_log(rng, 20_000, 4_000_000), k=_log(rng, 1, 32))
    if kind == "subset":
        n = _log(rng, 100_000, 5_000_000)
        return dict(c, n=n, queries=max(64, int(n * rng.uniform(0.02, 0.4))), k=_log(rng, 1, 128))
    if kind == "knn":
        return dict(c, n=_log(rng, 50_000, 5_000_000), queries=_log(rng, 100, 500_000),
                    k=_log(rng, 1, 200))
    if kind == "csr":
        # radii from each particle's own neighbours: floating-point snapshots
        c["coord"] = "f64"
        return dict(c, n=_log(rng, 50_000, 2_000_000))
    return dict(c, n=_log(rng, 100_000, 4_000_000), queries=_log(rng, 1000, 300_000),
                cap=rng.choice([16, 32, 64, 100]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
class _View:
    def __init__(self, ptr, n, typestr, owner):
        self.owner = owner  # a tensor over this view keeps the memory alive
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 2}


def _view(ptr, n, dtype, owner):
    """A tensor over n values of device memory that a framework object owns."""
    name = {torch.float32: "<f4", torch.float64: "<f8", torch.int32: "<i4", torch.int64: "<i8",
            torch.int8: "|i1"}[dtype]
    return torch.as_tensor(_View(ptr, n, name, owner), device="cuda")


def _device(t, coord=None):
    """The values of a tensor as a DeviceArray (unsigned where `coord` is an integer type)."""
    dt = ft.COORD_DTYPES[COORDS[coord]] if coord else \
        {torch.float32: np.float32, torch.float64: np.float64, torch.int32: np.int32,
         torch.int64: np.int64, torch.int8: np.int8}[t.dtype]
    a = ft.DeviceArray(t.numel(), dt)
    _view(a.ptr, t.numel(), t.dtype, a).copy_(t)
    return a


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(n, g):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _nfw(n, g):
    """Clustered positions in [0, BOX)^3, float64 (3, n)."""
    inside = int(round(0.7 * n))
    halos = max(4, int(round(inside / 3500.0)))
    mass = (1.0 + _rand(halos, g) * (1000.0 ** -0.9 - 1.0)) ** (1.0 / -0.9)
    conc = 4.0 + 8.0 * _rand(halos, g)
    centre = _rand(3 * halos, g).view(3, halos) * BOX
    rvir = 0.02 * BOX * (mass / 1000.0) ** (1.0 / 3.0)
    edges = torch.cumsum(mass, 0) / mass.sum()
    at = (torch.arange(inside, device="cuda", dtype=torch.float64) + 0.5) / max(inside, 1)
    h = torch.searchsorted(edges, at).clamp_(max=halos - 1)
    c = conc[h]
    u = _rand(inside, g) * (torch.log1p(c) - c / (1.0 + c))
    lo, hi = torch.zeros_like(u), c.clone()
    for _ in range(40):  # enclosed mass m(x) = ln(1 + x) - x / (1 + x) inverted by bisection
        mid = 0.5 * (lo + hi)
        below = torch.log1p(mid) - mid / (1.0 + mid) < u
        lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
    r = 0.5 * (lo + hi) * (rvir[h] / c)
    cos = 2.0 * _rand(inside, g) - 1.0
    phi = 2.0 * math.pi * _rand(inside, g)
    sin = torch.sqrt((1.0 - cos * cos).clamp_(min=0.0))
    out = torch.empty(3, n, device="cuda", dtype=torch.float64)
    for d, way in enumerate((sin * torch.cos(phi), sin * torch.sin(phi), cos)):
        out[d, :inside] = torch.remainder(centre[d][h] + r * way, BOX)
        out[d, inside:] = _rand(n - inside, g) * BOX
    out[out >= BOX] = 0.0
    return out  # halo by halo, then the background, as halo catalogues order them


def _positions(case, n, g):
    """Positions (3, n) in the case's coordinate type (integers as signed bit patterns)."""
    p = _nfw(n, g) if case["points"] == "clustered" else _rand(3 * n, g).view(3, n) * BOX
    return _as_coord(p, case)


def _as_coord(p, case):
    if case["coord"] in ("i32", "i64"):
        top = (1 << BITS) - 1
        return torch.floor(p / BOX * float(1 << BITS)).clamp_(0, top).to(TORCH[case["coord"]])
    return p.to(TORCH[case["coord"]])


def _config(case):
    fp = case["coord"] in ("f32", "f64")
    return ft.Config(sfc=CURVES[case["curve"]], bits_per_dim=case["bits"],
                     periodic=case["periodic"], box_length=BOX if fp and case["periodic"] else 0.0)


def _tree(case, n, pos, scratch=None):
    xyz = [_device(pos[d].contiguous(), case["coord"]) for d in range(3)]
    tree = ft.TreeSoA(n, COORDS[case["coord"]], _config(case))
    ft.build_bvh(ft.particles(*xyz), tree, scratch=scratch)
    return tree, xyz


def _tree_views(tree, case, n):
    """The arrays that a build writes, as tensors."""
    t, m = TORCH[case["coord"]], 2 * n - 1
    out = {a: _view(getattr(tree.c, a), m, t, tree)
           for a in ("min_x", "max_x", "min_y", "max_y", "min_z", "max_z")}
    for a in ("left_child", "right_child", "range_first", "range_last"):
        out[a] = _view(getattr(tree.c, a), n - 1, torch.int32, tree)
    out["parent"] = _view(tree.c.parent, m, torch.int32, tree)
    for a in ("id", "orig_idx"):
        out[a] = _view(getattr(tree.c, a), m, torch.int32, tree)[n - 1:]
    out["is_ghost"] = _view(tree.c.is_ghost, m, torch.int8, tree)[n - 1:]
    out["sorted_keys"] = _view(tree.c.sorted_keys, n, torch.int64, tree)
    return out


def _outputs(case, rows):
    fp = case["coord"] in ("f32", "f64")
    return {"index": torch.empty(rows, device="cuda", dtype=torch.int64),
            "d2": torch.empty(rows, device="cuda", dtype=torch.float64 if fp else torch.int64)}


def _probes(case, pos, q, g):
    """q points that follow the tree's density: a particle displaced by a
    Gaussian of a thousandth of the box."""
    n = pos.shape[1]
    pick = torch.randint(0, n, (q,), generator=g, device="cuda")
    step = torch.randn(3, q, generator=g, device="cuda", dtype=torch.float64) * (BOX / 1000.0)
    unit = BOX / float(1 << BITS) if case["coord"] in ("i32", "i64") else 1.0
    p = pos[:, pick].to(torch.float64) * unit + step
    p = torch.remainder(p, BOX) if case["periodic"] else p.clamp_(0.0, BOX * (1.0 - 2.0 ** -24))
    p[p >= BOX] = 0.0
    return _as_coord(p, case)


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind == "grad":
        return _prepare_grad(case, g, seed)
    if kind == "batch":
        return _prepare_batch(case, g)
    n = case["n"]
    pos = _positions(case, n, g)
    if kind in ("build", "step"):
        # a program keeps its tree and the build's work buffers from step to step
        xyz = [_device(pos[d].contiguous(), case["coord"]) for d in range(3)]
        ids = ghost = None
        if case.get("ids"):
            ids = _device(torch.randperm(n, generator=g, device="cuda").to(torch.int32))
            ghost = _device((torch.rand(n, generator=g, device="cuda") < 0.1).to(torch.int8))
        tree = ft.TreeSoA(n, COORDS[case["coord"]], _config(case))
        s = {"kind": kind, "tree": tree, "scratch": ft.BvhScratch(),
             "p": ft.particles(*xyz, id=ids, is_ghost=ghost),
             "views": _tree_views(tree, case, n)}
        if kind == "step":
            s.update(k=case["k"], out=_outputs(case, n * case["k"]))
        return s
    tree, _ = _tree(case, n, pos)
    s = {"kind": kind, "tree": tree, "k": case.get("k")}
    if kind == "self":
        s["out"] = _outputs(case, n * case["k"])
    elif kind == "subset":
        pick = torch.randperm(n, generator=g, device="cuda")[:case["queries"]]
        s["ids"] = _device(pick.to(torch.int32))
        s["out"] = _outputs(case, case["queries"] * case["k"])
    elif kind == "knn":
        q = _probes(case, pos, case["queries"], g)
        s["q"] = [_device(q[d].contiguous(), case["coord"]) for d in range(3)]
        s["out"] = _outputs(case, case["queries"] * case["k"])
    elif kind == "range":
        nq = case["queries"]
        q = _probes(case, pos, nq, g)
        s["q"] = [_device(q[d].contiguous(), case["coord"]) for d in range(3)]
        link = 0.2 * BOX / n ** (1.0 / 3.0)
        if case["coord"] in ("i32", "i64"):
            link = round(link / BOX * float(1 << BITS))
        r = torch.full((nq,), link, device="cuda", dtype=torch.float64).to(TORCH[case["coord"]])
        s["r"] = [_device(torch.zeros_like(r), case["coord"]), _device(r, case["coord"])]
        s["cap"] = case["cap"]
        # entries past a row's count are not written
        s["rows"] = torch.full((nq * case["cap"],), -1, device="cuda", dtype=torch.int32)
        s["counts"] = torch.empty(nq, device="cuda", dtype=torch.int32)
    elif kind == "csr":
        d2 = torch.empty(n * 32, device="cuda", dtype=torch.float64)
        ix = torch.empty(n * 32, device="cuda", dtype=torch.int64)
        ft.self_knn_query(tree, 32, results=ix.data_ptr(), dists=d2.data_ptr())
        h = 1.2 * torch.sqrt(d2.view(n, 32)[:, 31])
        s["q"] = [_device(_view(p, 2 * n - 1, torch.float64, tree)[n - 1:])
                  for p in (tree.c.min_x, tree.c.min_y, tree.c.min_z)]
        s["r"] = [_device(torch.zeros_like(h)), _device(h)]
        # a program keeps its offset and column buffers and grows the columns
        # when a step needs more; entries past the last hit are not written
        s["rows"] = torch.empty(n + 1, device="cuda", dtype=torch.int64)
        s["cols"] = torch.full((96 * n,), -1, device="cuda", dtype=torch.int32)
        s["n"] = n
    return s


def _prepare_batch(case, g):
    ct, nt = COORDS[case["coord"]], case["trees"]
    sizes = [int(round(case["n_min"] * (case["n_max"] / case["n_min"]) ** (t / max(nt - 1, 1))))
             for t in range(nt)]
    ks = (1, 8, 32, 128)
    trees, parts, nq, kk, of, qs = [], [], [], [], [], []
    for t, n in enumerate(sizes):
        pos = _positions(case, n, g)
        parts.append(tuple(_device(pos[d].contiguous(), case["coord"]) for d in range(3)))
        trees.append(ft.TreeSoA(n, ct, _config(case)))
        for r in range(2):
            m = max(1, int(case["queries"] / (2 * nt) * (0.4 + 1.2 * ((3 * t + 5 * r) % 7) / 6)))
            nq.append(m)
            kk.append(ks[(t + 2 * r + t // 4) % 4])
            of.append(t)
            qs.append(_probes(case, pos, m, g))
    reqs, _, rows = plan_requests(nq, kk, of)
    q = torch.cat(qs, dim=1)
    dq = [_device(q[d].contiguous(), case["coord"]) for d in range(3)]
    res, dst = ft.DeviceArray(rows, np.uint64), ft.DeviceArray(rows, np.uint64)
    b = Batch(ct)
    b.set_trees(trees, parts)
    b.set_queries(reqs, *dq, res, dst)
    # settings that a program has kept from an earlier tuning of its workload
    for c in range(4):
        b.set_tier(c, 0, "packet-reg1", 64, 16)
        b.set_tier(c, 2, "packet-reg8", 64, 32)
        b.set_tier(c, 4, "packet-reg32", 64, 16)
        b.set_tier(c, 6, "wave-merge128", 32, 8)
    b.run()
    b.capture()
    return {"kind": "batch", "batch": b, "trees": trees, "parts": parts, "q": dq,
            "out": {"index": _view(res.ptr, rows, torch.int64, res),
                    "d2": _view(dst.ptr, rows, torch.int64, dst)}}


def _features(case, g):
    """Feature rows and targets with the scales that snapshots give, float32."""
    rows = case["rows"]
    f = torch.zeros(rows, NF, device="cuda", dtype=torch.float64)
    depth = torch.randn(rows, generator=g, device="cuda", dtype=torch.float64)
    for j in range(4):
        f[:, j] = 24.0 + 2.0 * j + 3.0 * depth
        f[:, 4 + j] = 2.0 * (j + 1) * 0.69 + 0.4 * depth
    f[:, 8] = math.log(32.0)
    for j in range(9, 12):
        f[:, j] = 14.0 + 2.0 * depth
    noise = torch.randn(rows, 12, generator=g, device="cuda", dtype=torch.float64)
    f[:, :8] += 0.5 * noise[:, :8]
    f[:, 9:12] += noise[:, 9:12]
    y = 0.6 * f[:, 0] + 0.1 * f[:, 10] - 1.0 + 0.3 * noise[:, 8]
    return f.to(torch.float32), y.to(torch.float32)


def _norm(f, y):
    mu, sd = f.double().mean(0), f.double().std(0, unbiased=False)
    inv = torch.where(sd > 1e-6, 1.0 / sd.clamp(min=1e-6), torch.zeros_like(sd))
    mu[12:], inv[12:] = 0.0, 0.0
    tail = torch.stack([y.double().mean(), y.double().std(unbiased=False)])
    return torch.cat([mu, inv, tail]).to(torch.float32)


def _prepare_grad(case, g, seed):
    f, y = _features(case, g)
    m = MLP(init_params(seed), _norm(f, y).cpu().numpy(), 0.0)
    grad, loss = ft.DeviceArray(NPARAM + 16, np.float32), ft.DeviceArray(1, np.float32)
    return {"kind": "grad", "m": m, "f": _device(f.reshape(-1)), "y": _device(y),
            "rows": case["rows"], "g": grad, "l": loss,
            "out": {"grad": _view(grad.ptr, NPARAM, torch.float32, grad),
                    "loss": _view(loss.ptr, 1, torch.float32, loss)}}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "build":
        ft.build_bvh(s["p"], s["tree"], scratch=s["scratch"])
        return s["views"]
    if kind == "step":
        ft.build_bvh(s["p"], s["tree"], scratch=s["scratch"])
        ft.self_knn_query(s["tree"], s["k"], results=s["out"]["index"].data_ptr(),
                          dists=s["out"]["d2"].data_ptr())
        return {**s["out"], "tree": s["views"]}
    if kind == "self":
        ft.self_knn_query(s["tree"], s["k"], results=s["out"]["index"].data_ptr(),
                          dists=s["out"]["d2"].data_ptr())
        return s["out"]
    if kind == "subset":
        ft.self_knn_query_subset(s["tree"], s["ids"], s["k"],
                                 results=s["out"]["index"].data_ptr(),
                                 dists=s["out"]["d2"].data_ptr())
        return s["out"]
    if kind == "knn":
        ft.knn_query(s["tree"], *s["q"], s["k"], results=s["out"]["index"].data_ptr(),
                     dists=s["out"]["d2"].data_ptr())
        return s["out"]
    if kind == "range":
        ft.range_query(s["tree"], *s["q"], *s["r"], s["cap"], results=s["rows"].data_ptr(),
                       result_counts=s["counts"].data_ptr())
        return {"rows": s["rows"], "counts": s["counts"]}
    if kind == "csr":
        # counts and offsets, room for that many columns, then the list
        n, lib, rows = s["n"], ft.lib(), s["rows"]
        args = [ft.C.byref(s["tree"].c), *(a.ptr for a in s["q"]), *(a.ptr for a in s["r"]), n]
        _ok(lib.ft_range_query_csr(None, *args, rows.data_ptr(), None, 0))
        total = int(rows[n].item())
        if total > s["cols"].numel():
            s["cols"] = torch.full((total,), -1, device="cuda", dtype=torch.int32)
        _ok(lib.ft_range_query_csr(None, *args, rows.data_ptr(), s["cols"].data_ptr(), total))
        return {"rows": rows, "cols": s["cols"]}
    if kind == "batch":
        s["batch"].launch()
        return s["out"]
    _ok(ft.lib().ft_mlp_grad(None, s["m"].h, s["f"].ptr, s["y"].ptr, s["rows"], s["g"].ptr,
                             s["l"].ptr))
    return s["out"]


def _ok(rc):
    if rc:
        raise RuntimeError(ft.lib().ft_last_error().decode(errors="replace"))


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _knn_work(n, q, k, s, external):
    """Each query's answer written, its point read, and each leaf read once (a
    few queries need no more leaves than they return); a distance is 8
    operations."""
    touched = min(n, q * k)
    return {"bytes": q * 16.0 * k + touched * 3.0 * s + (q * 3.0 * s if external else 0.0),
            "flops": 8.0 * q * k}


def _build_work(n, s, ids):
    """The points (and ids and ghost flags) read; six box arrays over 2n nodes,
    child links, leaf ranges, parents, ids, flags, permutation and keys written."""
    read = n * (3.0 * s + (5.0 if ids else 0.0))
    return {"bytes": read + 12.0 * s * n + 16.0 * n + 8.0 * n + 9.0 * n + 8.0 * n, "flops": 0.0}


def work(case):
    kind = case["kind"]
    if kind == "grad":
        r = float(case["rows"])
        return {"bytes": r * 4.0 * (NF + 1) + 8.0 * NPARAM,
                "flops": r * 6.0 * (NF * 64 + 2 * 64 * 64 + 64)}
    s = float(SIZES[case["coord"]])
    if kind == "batch":
        nt = case["trees"]
        n = sum(case["n_min"] * (case["n_max"] / case["n_min"]) ** (t / max(nt - 1, 1))
                for t in range(nt))
        a, b = _build_work(n, s, False), _knn_work(n, case["queries"], 42, s, True)
        return {x: a[x] + b[x] for x in a}
    n = float(case["n"])
    if kind == "build":
        return _build_work(n, s, case["ids"])
    if kind == "step":
        a, b = _build_work(n, s, False), _knn_work(n, n, case["k"], s, False)
        return {x: a[x] + b[x] for x in a}
    if kind == "self":
        return _knn_work(n, n, case["k"], s, False)
    if kind in ("subset", "knn"):
        w = _knn_work(n, case["queries"], case["k"], s, kind == "knn")
        return {"bytes": w["bytes"] + (4.0 * case["queries"] if kind == "subset" else 0.0),
                "flops": w["flops"]}
    if kind == "csr":
        hits = 58.0  # 1.2^3 times 33, about
        return {"bytes": n * (5.0 * s + 3.0 * s + 8.0 + 4.0 * hits), "flops": 8.0 * n * hits}
    q, hits = float(case["queries"]), 0.5 * case["cap"]
    return {"bytes": q * (5.0 * s + 4.0 + 4.0 * hits) + min(n, q * hits) * 3.0 * s,
            "flops": 8.0 * q * hits}


# ---------------------------------------------------------------------------
# The outputs in 64 bits, by plain tensor code
# ---------------------------------------------------------------------------
def _morton_order(p, bits):
    """The stable order of Morton keys: each axis scaled to its extent, the top
    `bits` mantissa bits of 1 + x, interleaved with x lowest."""
    key = torch.zeros(p.shape[1], device=p.device, dtype=torch.int64)
    for a in range(3):
        lo, hi = p[a].min(), p[a].max()
        t = ((p[a] - lo) * (1.0 / (hi - lo))).clamp(0.0, 1.0 - 2.0 ** -53)
        v = ((1.0 + t).view(torch.int64) & ((1 << 52) - 1)) >> (52 - bits)
        for b in range(bits):
            key |= ((v >> b) & 1) << (3 * b + a)
    return torch.sort(key, stable=True)[1]


def _distances(pts, rows, k, period, skip):
    """The k smallest squared distances from each of `rows` (3, m) to pts (3, n)."""
    n, m, out = pts.shape[1], rows.shape[1], []
    step = max(1, 200_000_000 // n)
    for i in range(0, m, step):
        d2 = None
        for a in range(3):
            d = (rows[a, i:i + step, None] - pts[a][None, :]).abs()
            if period:
                d = torch.minimum(d, period - d)
            d2 = d * d if d2 is None else d2 + d * d
        if skip is not None:
            j = torch.arange(i, min(i + step, m), device=pts.device)
            d2[j - i, skip[j]] = float("inf")
        out.append(torch.topk(d2, k, dim=1, largest=False, sorted=True)[0])
    return torch.cat(out).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "grad":
        return _exact_grad(case, seed)
    if case["coord"] not in ("f32", "f64"):
        return None
    n = case["n"]
    if kind == "knn" and n * case["queries"] <= 30_000_000_000:
        g = _gen(seed)
        pos = _positions(case, n, g)
        q = _probes(case, pos, case["queries"], g)
        k = min(case["k"], n)
        return {"index": None, "d2": _distances(pos.double(), q.double(), k,
                                                BOX if case["periodic"] else None, None)}
    if kind in ("step", "self") and case["curve"] == "morton" and case["coord"] == "f64" \
            and n * n <= 30_000_000_000:
        pos = _positions(case, n, _gen(seed))
        pts = pos[:, _morton_order(pos, case["bits"])]
        own = torch.arange(n, device="cuda")
        d2 = _distances(pts, pts, case["k"], BOX if case["periodic"] else None, own)
        return {"index": None, "d2": d2} if kind == "self" else \
            {"index": None, "d2": d2, "tree": None}
    return None


def _exact_grad(case, seed):
    f, y = _features(case, _gen(seed))
    norm = _norm(f, y).double()
    p = torch.from_numpy(init_params(seed)).cuda().double()
    at, w = 0, []
    for shape in ((NF, 64), (64,), (64, 64), (64,), (64, 64), (64,), (64,), (1,)):
        size = math.prod(shape)
        w.append(p[at:at + size].view(shape))
        at += size
    x = (f.double() - norm[:NF]) * norm[NF:2 * NF]
    z1 = x @ w[0] + w[1]
    a1 = z1.clamp(min=0.0)
    z2 = a1 @ w[2] + w[3]
    a2 = z2.clamp(min=0.0)
    z3 = a2 @ w[4] + w[5]
    a3 = z3.clamp(min=0.0)
    e = (a3 @ w[6] + w[7]) - (y.double() - norm[2 * NF]) / norm[2 * NF + 1]
    do = 2.0 * e / e.numel()
    d3 = torch.outer(do, w[6]) * (z3 > 0)
    d2 = (d3 @ w[4].t()) * (z2 > 0)
    d1 = (d2 @ w[2].t()) * (z1 > 0)
    parts = [x.t() @ d1, d1.sum(0), a1.t() @ d2, d2.sum(0), a2.t() @ d3, d3.sum(0), a3.t() @ do,
             do.sum().view(1), torch.zeros(NPARAM - at, device="cuda", dtype=torch.float64)]
    return {"grad": torch.cat([v.reshape(-1) for v in parts]), "loss": (e * e).mean().view(1)}
