"""GPU kernels at the edges of their tiles and grids, against plain numpy or the
oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# 256 points per partial, at most 1,024 partials, 256 threads in the final block
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 65_536, 65_537, 262_144, 262_145, 1_000_003])
@pytest.mark.parametrize("ct", [O.CT_F32, O.CT_F64, O.CT_U32, O.CT_U64])
def test_bbox_reduction_sizes(ft, n, ct):
    rng = np.random.default_rng(n)
    p = [(rng.normal(size=n) * 1e3 + (0 if ct in (O.CT_F32, O.CT_F64) else 1e5))
         .astype(O.COORD_DTYPES[ct]) for _ in range(3)]
    # the extremes sit at the ends and in the last, partly filled stride
    p[0][n - 1] = p[0].max() + 1
    p[2][n // 2] = p[2].min()
    want = [f(a) for a in p for f in (np.min, np.max)]
    got = ft.compute_bbox(*p)  # host arrays: staged
    assert np.array_equal(got, np.array(want, O.COORD_DTYPES[ct]))


# 1,024 threads a block, at most 512 blocks: one partial block, whole blocks,
# one point more than the grid covers in one stride
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 524_288, 524_289])
def test_build_histogram_grid(ft, orc, n):
    rng = np.random.default_rng(n)
    x, y, z = (rng.integers(0, 1 << 21, n).astype(np.uint32) for _ in range(3))
    tree = ft.TreeSoA(n, O.CT_U32, ft.Config(sfc=O.SFC_PH, bits_per_dim=21))
    ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(a) for a in (x, y, z))), tree)
    keys = O.encode(O.CT_U32, O.SFC_PH, 21, x, y, z, None)
    order = np.argsort(keys, kind="stable")
    got = tree.to_host()
    assert np.array_equal(got["sorted_keys"], keys[order])
    assert np.array_equal(got["orig_idx"][n - 1:], order.astype(np.int32))


# 16 samples a tile, 8 waves a block, 256 blocks: part of a tile, a tile and one
# sample, a block and one tile, more tiles than waves (a wave takes two)
@pytest.mark.parametrize("n", [1, 15, 16, 17, 128, 129, 4096, 32_768, 32_785, 65_537])
def test_gradient_sample_counts(ft, n):
    """Against the float64 oracle with the same bf16 roundings.  The products'
    operands agree exactly up to activations that fall on the other side of a
    bf16 rounding step (2^-9 relative, a few of them per sum), so the gradient
    is held to 1 % of its largest component and the loss to 1e-3."""
    from fasttree_amd import learned as L
    from oracle import mlp as M

    rng = np.random.default_rng(n)
    f = np.zeros((n, 16), np.float32)
    f[:, :12] = rng.normal(size=(n, 12)) * 3 + 5
    y = (f[:, 0] * 0.5 + rng.normal(size=n)).astype(np.float32)
    p = L.init_params(n)
    p[9408:9472] *= 10  # an output layer whose gradient reaches the lower layers
    norm = L.norm_from(f, y) if n > 1 else L.default_norm()
    m = L.MLP(p, norm, 0.0)
    g, loss = m.grad(ft.DeviceArray.from_host(f.ravel()), ft.DeviceArray.from_host(y), n)
    el, eg = M.loss_and_grad(p, norm.astype(np.float64), f, y, rounding=True)
    assert abs(loss - el) <= 1e-3 * el + 1e-7
    assert np.abs(g - eg).max() <= 1e-2 * np.abs(eg).max()
    assert not g[9473:].any()


# 64 queries a packet: slots left by whole, partial and several packets, appended
# by one atomic per wave; all, some or none of the seeds too small
@pytest.mark.parametrize("n", [2, 63, 64, 65, 129, 4097])
@pytest.mark.parametrize("ct", [O.CT_U32, O.CT_F64])
@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
def test_slots_left_to_the_listed_pass(ft, orc, n, ct, share):
    rng = np.random.default_rng(n)
    fp = ct == O.CT_F64
    pts = [rng.integers(0, 1 << 20, n).astype(O.COORD_DTYPES[ct]) for _ in range(3)]
    k = min(8, n - 1)
    tree = ft.TreeSoA(n, ct, ft.Config(sfc=O.SFC_PH, bits_per_dim=21))
    ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(a) for a in pts)), tree)
    t = O.build_bvh(ct, *pts, sfc=O.SFC_PH, bits=21)
    rb, db = O.knn_bruteforce(t, k, True)
    small = rng.random(n) < share
    seed = np.where(small, 0, np.finfo(np.float64).max if fp else (1 << 60))
    seed = seed.astype(np.float64 if fp else np.uint64)
    stats = ft.DeviceArray(8, np.uint64).zero()
    r, d = ft.self_knn_query(tree, k, seed_bound=ft.DeviceArray.from_host(seed), stats=stats)
    assert np.array_equal(r, rb) and np.array_equal(d, db)
    assert stats.to_host()[3] == int(np.sum(seed < db[:, -1]))


def _doubles(name, n, seed):
    i = np.arange(n)
    rng = np.random.default_rng(seed)
    if name == "grid":  # distances exactly equal
        return [(i // 225).astype(float), (i // 15 % 15).astype(float), (i % 15).astype(float)]
    if name == "rounded grid":  # equal but for the last bits
        return [(i // 225) * 0.1 + 0.05, (i // 15 % 15) * 0.1 + 0.05, (i % 15) * 0.1 + 0.05]
    if name == "coincident":
        return [np.repeat(rng.random(-(-n // 8)), 8)[:n] for _ in range(3)]
    return [rng.random(n) ** 3 for _ in range(3)]


# list widths 4, 8, 16, 32 and passes of 32, full and not; packets of ties
# beside packets without
@pytest.mark.parametrize("k", [2, 4, 5, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("name", ["grid", "rounded grid", "coincident", "continuous"])
@pytest.mark.parametrize("ct", [O.CT_F64, O.CT_F32])
def test_packed_distances_of_floating_point(ft, orc, k, name, ct):
    n = 3375
    pts = [a.astype(O.COORD_DTYPES[ct]) for a in _doubles(name, n, k)]
    if name == "rounded grid":
        half = [a.astype(O.COORD_DTYPES[ct]) for a in _doubles("continuous", n, k + 1)]
        pts = [np.concatenate([a, b + a.max()]) for a, b in zip(pts, half)]
    n = len(pts[0])
    ids = np.random.default_rng(k).permutation(n)[: n // 4].astype(np.int32)
    for periodic, orig in ((0, False), (1, True)):
        box = float(max(a.max() for a in pts)) * 1.01 if periodic else 0.0
        tree = ft.TreeSoA(n, ct, ft.Config(sfc=O.SFC_PH, bits_per_dim=21, periodic=periodic,
                                           box_length=box, return_orig_indices=orig))
        ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(a) for a in pts)), tree)
        t = O.build_bvh(ct, *pts, sfc=O.SFC_PH, bits=21, periodic=periodic, box=box,
                        orig_indices=int(orig))
        rb, db = O.knn_bruteforce(t, k, True)
        r, d = ft.self_knn_query(tree, k, max_k=64, algorithm=ft.ALGO_PACKET)
        assert np.array_equal(d, db) and np.array_equal(r, rb)
        r, d = ft.self_knn_query_subset(tree, ids, k, algorithm=ft.ALGO_PACKET)
        assert np.array_equal(d, db[ids]) and np.array_equal(r, rb[ids])


def test_packed_distances_that_overflow(ft, orc):
    """Squared distances beyond the coordinate type's range are no neighbours;
    huge finite ones are."""
    for ct, big in ((O.CT_F64, 1e160), (O.CT_F32, 1e19)):
        rng = np.random.default_rng(5)
        pts = [(rng.random(200) * 1e-3 * big).astype(O.COORD_DTYPES[ct]) for _ in range(3)]
        for a in pts:
            a[100:] += np.array(big * 30, a.dtype)  # d2 to the other half overflows
        tree = ft.TreeSoA(200, ct, ft.Config(sfc=O.SFC_PH, bits_per_dim=21))
        ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(a) for a in pts)), tree)
        for k in (8, 32):
            want = ft.self_knn_query(tree, k, algorithm=ft.ALGO_PLAIN)
            got = ft.self_knn_query(tree, k, algorithm=ft.ALGO_PACKET)
            for a, b in zip(got, want):
                assert np.array_equal(a, b)


# The automatic choice on either side of its lines: few queries (a wave each,
# unsorted up to 24,576), packets of 32 and 64, packets handed over
@pytest.mark.parametrize("n,nq", [(3000, 1), (3000, 64), (3000, 65), (40_000, 24_576),
                                  (40_000, 24_577), (3000, 40_000), (3000, 160_000)])
@pytest.mark.parametrize("ct,k", [(O.CT_U64, 8), (O.CT_F64, 16), (O.CT_F32, 1), (O.CT_U32, 33)])
def test_automatic_external_queries(ft, orc, n, nq, ct, k):
    rng = np.random.default_rng(nq + k)
    fp = ct in (O.CT_F32, O.CT_F64)
    hi = 1.0 if fp else float(1 << 21)
    p = rng.random((3, n)) ** 4 * hi  # dense near the origin: packets far out are wide
    q = np.concatenate([rng.random((3, nq - nq // 2)) ** 4, rng.random((3, nq // 2))], 1) * hi
    pts = [a.astype(O.COORD_DTYPES[ct]) for a in p]
    qs = [np.ascontiguousarray(a[rng.permutation(nq)].astype(O.COORD_DTYPES[ct])) for a in q]
    tree = ft.TreeSoA(n, ct, ft.Config(sfc=O.SFC_PH, bits_per_dim=21))
    ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(a) for a in pts)), tree)
    t = O.build_bvh(ct, *pts, sfc=O.SFC_PH, bits=21)
    r, d = ft.knn_query(tree, *qs, k)
    rows = rng.choice(nq, min(nq, 300), replace=False)
    rb, db = O.knn_bruteforce(t, k, queries=[a[rows] for a in qs])
    assert np.array_equal(d[rows], db) and np.array_equal(r[rows], rb)
    w, wd = ft.knn_query(tree, *qs, k, algorithm=ft.ALGO_WAVE)
    assert np.array_equal(r, w) and np.array_equal(d, wd)


# 150,000 queries: packets of 32 below, 64 above; few queries below 900 * 1.7 *
# cbrt(n); the clustered half makes packets that pass their leaf limit
@pytest.mark.parametrize("n", [20_000, 60_000, 149_999, 150_001])
@pytest.mark.parametrize("ct,k", [(O.CT_U32, 8), (O.CT_F64, 32), (O.CT_F64, 64)])
def test_automatic_self_queries(ft, n, ct, k):
    rng = np.random.default_rng(n)
    hi = 1.0 if ct == O.CT_F64 else float(1 << 21)
    p = np.concatenate([rng.random((3, n // 2)), rng.random((3, n - n // 2)) ** 6], 1) * hi
    pts = [np.ascontiguousarray(a.astype(O.COORD_DTYPES[ct])) for a in p]
    tree = ft.TreeSoA(n, ct, ft.Config(sfc=O.SFC_MORTON, bits_per_dim=21))
    ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(a) for a in pts)), tree)
    r, d = ft.self_knn_query(tree, k, max_k=64)
    w, wd = ft.self_knn_query(tree, k, max_k=64, algorithm=ft.ALGO_WAVE)
    assert np.array_equal(r, w) and np.array_equal(d, wd)


# Range queries on both sides of the wave / packet line (400 * cbrt(n)), packets
# with and without an inner radius, queries too far apart for the relative
# filter, radii of zero, beyond the box and not a number, rows past the cap and
# past the CSR pool of 128
@pytest.mark.parametrize("n,nq", [(1, 70), (2, 5000), (64, 1700), (3000, 1), (3000, 5768),
                                  (3000, 5770), (30_000, 13_000)])
@pytest.mark.parametrize("ct", [O.CT_F64, O.CT_F32, O.CT_U64, O.CT_U32])
@pytest.mark.parametrize("periodic", [0, 1])
def test_range_queries_against_plain_distances(ft, n, nq, ct, periodic):
    rng = np.random.default_rng(n + nq)
    fp = ct in (O.CT_F64, O.CT_F32)
    side = 100.0 if fp else float(1 << 21)
    dt = O.COORD_DTYPES[ct]
    cast = (lambda a: a.astype(dt)) if fp else (lambda a: np.floor(a).astype(dt))
    pts = [cast(a) for a in rng.random((3, n)) ** 3 * side]
    q = [cast(a) for a in rng.random((3, nq)) ** 3 * side]
    r1 = rng.choice([0.0, 0.003, 0.02, 0.1, 0.3], nq) * side
    r0 = np.where(rng.random(nq) < 0.5, 0.0, r1 * rng.random(nq))
    r1, r0 = cast(r1), cast(r0)
    if fp and nq > 100:
        r1[3], r0[7], r1[11] = np.nan, np.nan, np.inf
    tree = ft.TreeSoA(n, ct, ft.Config(sfc=O.SFC_PH, bits_per_dim=21, periodic=periodic,
                                       box_length=side if fp and periodic else 0.0))
    ft.build_bvh(ft.particles(*(ft.DeviceArray.from_host(a) for a in pts)), tree)
    g = tree.to_host()
    x = [g[a][n - 1:] for a in ("min_x", "min_y", "min_z")]
    rows = np.arange(nq) if nq * n < 3e7 else np.unique(np.r_[3, 7, 11, rng.integers(0, nq, 600)])
    d2 = None
    for a in range(3):
        if fp:
            d = np.abs(q[a][rows, None] - x[a][None, :])
            d = np.minimum(d, dt(side) - d) if periodic else d
        else:
            d = q[a][rows, None].astype(np.int64) - x[a][None, :].astype(np.int64)
            if periodic:
                d = (d + (1 << 20)) % (1 << 21) - (1 << 20)
        d2 = d * d if d2 is None else d2 + d * d
    if fp:
        lo, hi = r0.astype(np.float64) ** 2, r1.astype(np.float64) ** 2
        d2 = d2.astype(np.float64)
    else:
        lo, hi = r0.astype(np.int64) ** 2, r1.astype(np.int64) ** 2
    hit = (d2 >= lo[rows, None]) & (d2 <= hi[rows, None])
    cap = 20
    res, counts = ft.range_query(tree, *q, r0, r1, cap)
    assert np.array_equal(counts[rows], hit.sum(1))
    rp, cols = ft.range_query_csr(tree, *q, r0, r1)
    assert np.array_equal(np.diff(rp), counts)
    for i, row in enumerate(rows):
        want = np.flatnonzero(hit[i])
        assert np.array_equal(cols[rp[row]:rp[row + 1]], want)
        assert np.array_equal(res[row][:min(cap, len(want))], want[:cap])
