"""Query kernels on inputs at the edges of what they accept: coordinates that are
not numbers, distances that overflow, trees deeper than a walk's stack, buffers
under capture, tied distances.  Against plain numpy or the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

FP = (O.CT_F64, O.CT_F32)


def build(ft, ct, pts, periodic=0, box=0.0, sfc=O.SFC_PH, orig=False):
    tree = ft.TreeSoA(len(pts[0]), ct, ft.Config(sfc=sfc, bits_per_dim=21, periodic=periodic,
                                                 box_length=box, return_orig_indices=orig))
    ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(np.ascontiguousarray(a)) for a in pts)),
                 tree)
    return tree


def leaves(tree):
    n = tree.num_leaves
    g = tree.to_host()
    return [g[a][n - 1:] for a in ("min_x", "min_y", "min_z")]


def squared(q, x, box=0.0):
    """The library's floating-point squared distances: one rounding an operation."""
    d2 = None
    with np.errstate(over="ignore"):
        for a in range(3):
            d = np.abs(q[a][:, None] - x[a][None, :])
            d = np.minimum(d, x[a].dtype.type(box) - d) if box else d
            d2 = d * d if d2 is None else d2 + d * d
    return d2.astype(np.float64)


def nearest(d2, k):
    """Canonical rows: (d2, index) ascending, finite distances only."""
    d2 = np.where(np.isfinite(d2), d2, np.inf)
    idx = np.argsort(d2, axis=1, kind="stable")[:, :k]
    d = np.take_along_axis(d2, idx, 1)
    none = ~np.isfinite(d)
    return (np.where(none, np.uint64(2**64 - 1), idx.astype(np.uint64)),
            np.where(none, -np.finfo(np.float64).max, d))


# 64 queries in the caller's order put a bad one into lanes 0 and 32; more are
# sorted along the curve, and a tenth of them bad reaches both lanes of some packet
@pytest.mark.parametrize("axes", [(0,), (1, 2), (0, 1, 2)])
@pytest.mark.parametrize("nq", [64, 6000])
@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("ct", FP)
def test_a_query_that_is_not_a_number_empties_its_own_row_only(ft, orc, ct, periodic, nq, axes):
    from fasttree_amd.batch import Batch, plan_requests
    dt = O.COORD_DTYPES[ct]
    rng = np.random.default_rng(nq + len(axes))
    n, box = 2000, 100.0
    pts = [(rng.random(n) * box).astype(dt) for _ in range(3)]
    q = [(rng.random(nq) * box).astype(dt) for _ in range(3)]
    bad = np.array([0, 32]) if nq == 64 else rng.choice(nq, nq // 10, replace=False)
    for a in axes:
        q[a][bad] = np.nan
    tree = build(ft, ct, pts, periodic, box if periodic else 0.0)
    d2 = squared(q, leaves(tree), box if periodic else 0.0)
    assert np.isnan(d2[bad]).all()
    r1 = rng.choice([3.0, 8.0, 15.0], nq).astype(dt)
    r0 = np.where(rng.random(nq) < 0.7, 0.0, 2.0).astype(dt)
    hit = (d2 >= r0[:, None].astype(float) ** 2) & (d2 <= r1[:, None].astype(float) ** 2)
    res, counts = ft.range_query(tree, *q, r0, r1, 40)
    rp, cols = ft.range_query_csr(tree, *q, r0, r1)
    assert np.array_equal(counts, hit.sum(1)) and np.array_equal(np.diff(rp), counts)
    assert np.array_equal(cols, np.nonzero(hit)[1])
    for i in range(nq):
        assert np.array_equal(res[i][:min(40, counts[i])], np.flatnonzero(hit[i])[:40])
    for k in (8, 32, 64):
        want, dist = nearest(d2, k)
        for algo in (ft.ALGO_PACKET, ft.ALGO_AUTO):
            if algo == ft.ALGO_AUTO and k > 32:
                continue  # the wave tier lists distances that are not numbers last
            r, d = ft.knn_query(tree, *q, k, algorithm=algo)
            good = np.setdiff1d(np.arange(nq), bad)
            assert np.array_equal(r[good], want[good]) and np.array_equal(d[good], dist[good])
            if algo == ft.ALGO_PACKET:
                assert (r[bad] == np.uint64(2**64 - 1)).all()
        if k <= 32:
            reqs, _, tr = plan_requests([nq], [k], [0])
            dq = [ft.DeviceArray.from_host(a) for a in q]
            r, d = ft.DeviceArray(tr, np.uint64), ft.DeviceArray(tr, np.float64)
            b = Batch(ct)
            b.set_trees([tree])
            b.set_queries(reqs, *dq, r, d)
            b.run()
            r, d = r.to_host().reshape(nq, k), d.to_host().reshape(nq, k)
            assert np.array_equal(r[good], want[good]) and np.array_equal(d[good], dist[good])


# Few queries (a wave each), many (packets, with and without a leaf limit), and
# above k = 32 the passes that the automatic choice takes instead of waves
@pytest.mark.parametrize("name", ["overflow", "not a number"])
@pytest.mark.parametrize("n,nq", [(200, 50), (200, 160_000), (3000, 200), (3000, 160_000)])
@pytest.mark.parametrize("ct", FP)
def test_distances_that_are_not_finite_do_not_depend_on_the_tier(ft, orc, ct, n, nq, name):
    dt = O.COORD_DTYPES[ct]
    rng = np.random.default_rng(n + nq)
    pts = [(rng.random(n) * 100).astype(dt) for _ in range(3)]
    if name == "overflow":  # five points whose distance to the others is infinite
        far = np.array(1e160 if ct == O.CT_F64 else 1e25, dt)
        for a in pts:
            a[n - 5:] += far
    else:  # five points with three coordinates each
        pts[1][5:] = np.nan
    tree = build(ft, ct, pts)
    x = leaves(tree)
    pick = rng.integers(0, n, nq)
    pick[:40] = np.flatnonzero(np.isfinite(x[1]) & (x[1] > 1000 if name == "overflow" else x[1] < 200))[
        rng.integers(0, 5, 40)]
    q = [np.ascontiguousarray(a[pick]) for a in x]
    rows = np.unique(np.r_[:40, rng.integers(0, nq, 300)])
    d2 = squared([a[rows] for a in q], x)
    ids = np.arange(n, dtype=np.int32)
    for k in (4, 8, 32):
        want, dist = nearest(d2, k)
        r, d = ft.knn_query(tree, *q, k)
        assert np.array_equal(r[rows], want) and np.array_equal(d[rows], dist)
        for call in (lambda **o: ft.self_knn_query(tree, k, **o),
                     lambda **o: ft.self_knn_query_subset(tree, ids, k, **o)):
            # (the per-lane tier tests a leaf as a box, which drops a NaN axis)
            tiers = [ft.ALGO_PACKET] + [ft.ALGO_PLAIN] * (name == "overflow")
            for a, b in ((call(), call(algorithm=t)) for t in tiers):
                assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    for k in (33, 64):  # the wave tier's rows: every point, those last
        for call in (lambda **o: ft.knn_query(tree, *q, k, **o),
                     lambda **o: ft.self_knn_query(tree, k, max_k=64, **o),
                     lambda **o: ft.self_knn_query_subset(tree, ids, k, **o)):
            a, b = call(), call(algorithm=ft.ALGO_WAVE)
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1], equal_nan=True)


# build_tree takes the original indices from its caller: any that an int32 holds
@pytest.mark.parametrize("base", [0, (1 << 30) - 250, (1 << 31) - 501])
@pytest.mark.parametrize("ct", FP)
def test_original_indices_of_any_size(ft, orc, ct, base):
    n, dt = 500, O.COORD_DTYPES[ct]
    rng = np.random.default_rng(3)
    pts = [(rng.random(n) * 100).astype(dt) for _ in range(3)]
    for a in pts:
        a[::5] = a[0]  # ties, ordered by the index
    cfg = ft.Config(sfc=O.SFC_MORTON, bits_per_dim=21, return_orig_indices=True)
    key = ft.sfc_encode(*pts, cfg, bbox=ft.compute_bbox(*pts))
    o = np.argsort(key, kind="stable")
    s = [np.ascontiguousarray(a[o]) for a in pts]
    orig = (rng.permutation(n) + base).astype(np.int32)
    tree = ft.TreeSoA(n, ct, cfg)
    dev = ft.DeviceArray.from_host
    ft.build_tree(tree, dev(key[o]), *(dev(a) for a in s), dev(np.arange(n, dtype=np.uint32)),
                  dev(np.zeros(n, np.int8)), dev(orig))
    d2 = squared(s, s)
    d2[np.arange(n), np.arange(n)] = np.inf
    col = np.argsort(orig)
    for k in (1, 4, 8, 16, 32, 64):
        want, dist = nearest(d2[:, col], k)
        want = orig[col][want.astype(np.int64)]
        for algo in (ft.ALGO_PACKET, ft.ALGO_AUTO):
            r, d = ft.self_knn_query(tree, k, max_k=64, algorithm=algo)
            assert np.array_equal(d, dist) and np.array_equal(r, want.astype(np.uint64))


# A first call on the stream is small; the second sizes the buffers and takes a
# wave per query (or leaves no slot); the captured one takes packets
@pytest.mark.parametrize("name", ["sorted waves", "unsorted waves", "float packets", "range"])
def test_buffers_fit_a_captured_call_of_another_tier(ft, orc, name):
    rng = np.random.default_rng(7)
    ct = O.CT_F32 if name == "float packets" else O.CT_U64
    dt = O.COORD_DTYPES[ct]
    pts = [rng.integers(0, 1 << 21, 200_000).astype(dt) for _ in range(3)]
    tree = build(ft, ct, pts)
    nq = {"sorted waves": 60_000, "unsorted waves": 20_000, "float packets": 170_000}.get(name, 20_000)
    q = [ft.DeviceArray.from_host(rng.integers(0, 1 << 21, nq).astype(dt)) for _ in range(3)]
    s = ft.Stream()
    if name == "range":
        few = build(ft, ct, [a[:300] for a in pts])  # 20,000 queries of 300 points: packets
        r = [ft.DeviceArray.from_host(np.full(nq, v, dt)) for v in (0, 200_000)]
        out = ft.DeviceArray(nq * 30, np.int32), ft.DeviceArray(nq, np.int32)
        call = lambda: ft.range_query(few, *q, *r, 30, *out, stream=s)
        warm = lambda: ft.range_query(tree, *q, *r, 30, *out, stream=s)
    else:
        out = ft.DeviceArray(nq * 32, np.uint64), ft.DeviceArray(nq * 32, ft.dist_dtype(ct))
        pk = ft.ALGO_PACKET
        call = lambda: ft.knn_query(tree, *q, 8, *out, stream=s, algorithm=pk)
        if name == "float packets":
            warm = lambda: ft.knn_query(tree, *q, 1, *out, stream=s, algorithm=ft.ALGO_WAVE)
        else:
            warm = lambda: ft.knn_query(tree, *q, 32 if name == "sorted waves" else 8, *out, stream=s)
    small = [ft.DeviceArray.from_host(rng.integers(0, 1 << 21, 300).astype(dt)) for _ in range(3)]
    tmp = ft.DeviceArray(2400, np.uint64), ft.DeviceArray(2400, ft.dist_dtype(ct))
    ft.knn_query(tree, *small, 8, *tmp, stream=s, algorithm=ft.ALGO_PACKET)
    warm()
    s.synchronize()
    with ft.Graph(s) as g:
        call()
    used = nq if name == "range" else nq * 8
    got = []
    for _ in range(3):
        for a in out:
            a.zero()
        g.launch()
        s.synchronize()
        got.append([a.to_host()[:used] for a in out])
    call()
    s.synchronize()
    want = [a.to_host()[:used] for a in out]
    for rows in got:
        assert np.array_equal(rows[1], want[1])
        assert name == "range" or np.array_equal(rows[0], want[0])


# Seeded queries whose distances tie: seeds that hold too few neighbours, the k-th
# distance itself and more, one lane beside the other
@pytest.mark.parametrize("k", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("name", ["grid", "rounded grid"])
@pytest.mark.parametrize("ct", FP)
def test_seeds_on_tied_distances(ft, orc, ct, name, k):
    i = np.arange(3375)
    pts = [(i // 225).astype(float), (i // 15 % 15).astype(float), (i % 15).astype(float)]
    if name == "rounded grid":  # equal but for the last bits
        pts = [a * 0.1 + 0.05 for a in pts]
    pts = [a.astype(O.COORD_DTYPES[ct]) for a in pts]
    side = 15.0 if name == "grid" else 1.5
    for periodic in (0, 1):
        tree = build(ft, ct, pts, periodic, side if periodic else 0.0)
        t = O.build_bvh(ct, *pts, sfc=O.SFC_PH, bits=21, periodic=periodic,
                        box=side if periodic else 0.0)
        rb, db = O.knn_bruteforce(t, k, True)
        rng = np.random.default_rng(k)
        for share in (0.0, 0.02, 0.4):  # of the seeds too small
            seed = db[:, -1] * rng.choice([1.0, 1.5, 4.0], len(i))
            seed = np.where(rng.random(len(i)) < share, db[:, k // 2] * 0.5, seed)
            r, d = ft.self_knn_query(tree, k, max_k=64, seed_bound=ft.DeviceArray.from_host(seed))
            assert np.array_equal(d, db) and np.array_equal(r, rb)


def list_shaped(ft, tree, order):
    """`tree` reshaped into a list: internal node i holds leaf i and node i + 1, its
    leaves in `order` -- a valid tree, as many levels deep as it has leaves."""
    n = tree.num_leaves
    ct = tree.coord_type
    cs, m, buf = np.dtype(O.COORD_DTYPES[ct]).itemsize, 2 * n - 1, bytearray(tree.serialize())
    sizes = [m * cs] * 6 + [(n - 1) * 4] * 2 + [m * 4, m * 4, m, m * 4, n * 8] + [(n - 1) * 4] * 2
    at = 64 + 16 + np.r_[0, np.cumsum(sizes)]
    view = lambda i, dt: np.frombuffer(buf, dt, sizes[i] // np.dtype(dt).itemsize, at[i])
    for a in range(6):
        c = view(a, O.COORD_DTYPES[ct])
        c[n - 1:] = c[n - 1:][order]
        acc = np.maximum if a % 2 else np.minimum
        c[:n - 1] = acc.accumulate(c[n - 1:][::-1])[::-1][:n - 1]
    i = np.arange(n - 1)
    left, right, parent = view(6, np.int32), view(7, np.int32), view(8, np.int32)
    left[:], right[:] = n - 1 + i, np.where(i + 1 < n - 1, i + 1, 2 * n - 2)
    parent[0], parent[left], parent[right] = -1, i, i
    view(13, np.int32)[:], view(14, np.int32)[:] = i, n - 1
    return ft.TreeSoA.deserialize(bytes(buf))


# A wave's stack holds 128 entries.  Lists of 64 to 1,024 neighbours; the leaves in
# random order, so that many more than 128 stay within the first bound
@pytest.mark.parametrize("k", [32, 64, 128, 200, 1000])
@pytest.mark.parametrize("ct", [O.CT_F64, O.CT_U32])
def test_trees_deeper_than_a_walk_s_stack(ft, orc, ct, k):
    rng = np.random.default_rng(k)
    n, nq, side = 3000, 100, 1000.0
    dt = O.COORD_DTYPES[ct]
    pts = [(rng.random(n) * side).astype(dt) for _ in range(3)]
    tree = list_shaped(ft, build(ft, ct, pts), rng.permutation(n))
    x = [a.astype(np.float64) for a in leaves(tree)]
    q = [(rng.random(nq) * side).astype(dt) for _ in range(3)]
    want, dist = nearest(squared([a.astype(np.float64) for a in q], x), k)
    r, d = ft.knn_query(tree, *q, k, max_k=1024)
    assert np.array_equal(d, dist) and np.array_equal(r, want)
    ids = rng.permutation(n)[:nq].astype(np.int32)
    d2 = squared([a[ids] for a in x], x)
    d2[np.arange(nq), ids] = np.inf
    want, dist = nearest(d2, k)
    r, d = ft.self_knn_query_subset(tree, ids, k, max_k=1024, algorithm=ft.ALGO_WAVE)
    assert np.array_equal(d, dist) and np.array_equal(r, want)


# Every query's neighbours are insertions of some pass, and a query is in [3] when
# the pass that answered it was the second: packets whose distances tie (whole or a
# few of their lanes), packets over their leaf limit, passes of 32
@pytest.mark.parametrize("k", [8, 32, 64])
@pytest.mark.parametrize("name", ["grid", "rounded grid", "half grid", "wide packets", "scattered"])
def test_counters_cover_the_second_pass(ft, orc, name, k):
    rng = np.random.default_rng(k)
    i = np.arange(24_389)
    pts = [(i // 841).astype(float), (i // 29 % 29).astype(float), (i % 29).astype(float)]
    if name != "grid":  # distances that agree but for their last bits
        pts = [a * 0.1 + 0.05 for a in pts]
    if name == "half grid":
        pts = [a + (i > 12_000) * rng.random(len(i)) * 0.3 for a in pts]
    if name in ("wide packets", "scattered"):
        pts = [rng.random(3000) ** 4 for _ in range(3)]
    tree = build(ft, O.CT_F64, pts)
    stats = ft.DeviceArray(8, np.uint64).zero()
    if name in ("wide packets", "scattered"):
        nq = 160_000
        q = [np.r_[rng.random(nq // 2) ** 4, rng.random(nq // 2)] for _ in range(3)]
        ft.knn_query(tree, *q, k, stats=stats,
                     algorithm=ft.ALGO_AUTO if name == "wide packets" else ft.ALGO_PACKET)
    else:
        nq = len(i)
        ft.self_knn_query(tree, k, max_k=64, algorithm=ft.ALGO_PACKET, stats=stats)
    st = stats.to_host()
    print(name, k, st)
    assert st[4] >= nq * k and st[1] * 64 >= nq * k and st[0] > 0
    assert st[3] <= nq
    if name == "rounded grid":
        assert st[3] > 0.9 * nq


def gridded(name, n, seed):
    """Doubles whose distances tie: on a grid that cut keys hold exactly, on one too
    fine for them, on a rounded one, and the first with single points off it."""
    rng = np.random.default_rng(seed)
    pts = [rng.integers(0, 16, n) / 16.0 for _ in range(3)]
    if name == "far from the origin":
        return [a + 2.0**30 for a in pts]
    if name == "too fine":  # distances differ far below the cut
        return [a + rng.integers(0, 2, n) * 2.0**-44 for a in pts]
    if name == "rounded":
        return [(a + 1 / 32) / 0.9999123 for a in pts]
    if name == "single points off":
        off = rng.choice(n, 5, replace=False)
        for a in pts:
            a[off] += 2.0**-44
    return pts


# Packets of 16, 32 and 64 (a quarter of their lanes makes them tied ones); with a
# fill, with none, in passes; equal distances ordered by rank and by original index
@pytest.mark.parametrize("width", [16, 32, 64])
@pytest.mark.parametrize("k", [3, 8, 20, 32, 40])
@pytest.mark.parametrize("name", ["exact", "far from the origin", "too fine", "rounded",
                                  "single points off"])
def test_tied_doubles_on_grids(ft, orc, name, k, width):
    n = 3000
    pts = gridded(name, n, k)
    rng = np.random.default_rng(k)
    ids = rng.permutation(n)[:1000].astype(np.int32)
    far = [np.r_[a[ids], a[ids[:300]] + 1 / 64] for a in pts]  # between the points too
    for periodic, orig, box in ((0, False, 0.0), (1, False, 2.0), (1, False, 1.0000001), (0, True, 0.0)):
        if periodic and name == "far from the origin":
            continue  # (a periodic box holds its points)
        if periodic and box < 1.01 and name == "rounded":
            box = 1.1
        tree = build(ft, O.CT_F64, pts, periodic, box, orig=orig)
        t = O.build_bvh(O.CT_F64, *pts, sfc=O.SFC_PH, bits=21, periodic=periodic, box=box,
                        orig_indices=int(orig))
        o = dict(algorithm=ft.ALGO_PACKET, group_width=width)
        rb, db = O.knn_bruteforce(t, k, True)
        r, d = ft.self_knn_query(tree, k, max_k=64, **o)
        assert np.array_equal(d, db) and np.array_equal(r, rb)
        r, d = ft.self_knn_query_subset(tree, ids, k, **o)
        assert np.array_equal(d, db[ids]) and np.array_equal(r, rb[ids])
        q = [np.mod(a, box) for a in far] if periodic else far
        rb, db = O.knn_bruteforce(t, k, queries=q)
        r, d = ft.knn_query(tree, *q, k, **o)
        assert np.array_equal(d, db) and np.array_equal(r, rb)


# 16 samples a tile, 8 waves a block, 256 blocks: the last sample, the first of its
# tile, and the edges of a tile, a block and the grid's first stride
@pytest.mark.parametrize("n", [1, 15, 17, 128, 129, 4096, 4113, 32_767, 32_785, 65_537])
def test_no_sample_of_a_gradient_is_lost_or_repeated(ft, n):
    """Targets are the network's own outputs but for a few marked samples, which
    carry the loss and the gradient.  Loss and gradient agree with the float64
    oracle to 1 % (activations on the other side of a bf16 step, 2^-9, shift an
    output by about as much; the marked residuals are 3 to 6 of the outputs'
    scale), and leaving out or doubling any one marked sample in the oracle moves
    both by more than twice that."""
    from fasttree_amd import learned as L
    from oracle import mlp as M

    rng = np.random.default_rng(n)
    f = np.zeros((n, 16), np.float32)
    f[:, :12] = rng.normal(size=(n, 12)) * 3 + 5
    p = L.init_params(n)
    p[9408:9472] *= 10
    norm = L.norm_from(f, f[:, 0] + rng.normal(size=n)) if n > 1 else L.default_norm()
    nd = norm.astype(np.float64)
    out, _ = M.forward(p, nd, f)
    scale = max(float(np.abs(out).max()), 1.0)
    marks = sorted({0, n - 1, (n - 1) // 16 * 16, max(n - 17, 0), min(15, n - 1), min(128, n - 1),
                    min(32_767, n - 1), min(32_768, n - 1)})
    e = np.zeros(n)
    e[marks] = scale * (3 + 3 * rng.random(len(marks)))
    y = ((out - e) * nd[33] + nd[32]).astype(np.float32)
    el, eg = M.loss_and_grad(p, nd, f[marks], y[marks])
    el, eg = el * len(marks) / n, eg * len(marks) / n
    top = np.abs(eg).max()
    for i, m in enumerate(marks):
        one, og = M.loss_and_grad(p, nd, f[m:m + 1], y[m:m + 1])
        assert one / n > 2e-2 * el and np.abs(og / n).max() > 2e-2 * top
    m = L.MLP(p, norm, 0.0)
    g, loss = m.grad(ft.DeviceArray.from_host(f.ravel()), ft.DeviceArray.from_host(y), n)
    assert abs(loss - el) <= 1e-2 * el
    assert np.abs(g - eg).max() <= 1e-2 * top
