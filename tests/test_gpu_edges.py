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
