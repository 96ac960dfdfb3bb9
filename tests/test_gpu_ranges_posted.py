"""Bounds read back: one set and arrays, value counts at the edges of what a thread, a block and the read-back by stores take,
to the bit (boxes of dyadic numbers have exact range sums)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


@pytest.mark.parametrize("N,count", [(1, 1), (1, 2), (127, 1), (128, 1), (129, 1), (255, 1), (256, 1), (257, 1), (10, 100), (3, 171),
                                     (1, 513), (2, 1024), (1000, 7), (4099, 5), (65536, 1), (64, 1024), (65537, 1), (65, 1024)])
def test_bounds_posted(nnv, N, count):
    rs = np.random.RandomState(7 * N + count)
    centre = rs.randint(-64, 64, (N, count)) / 32.0
    half = rs.randint(1, 1 << 12, (N, count)) / 1024.0
    lb, ub = np.asfortranarray(centre - half), np.asfortranarray(centre + half)
    if count == 1:
        glb, gub = (x[:, None] for x in nnv.Star(lb[:, 0], ub[:, 0]).estimateRanges())
    else:
        glb, gub = nnv.Star.estimateRanges_array(nnv.Star.from_boxes(lb, ub))
    assert np.array_equal(glb, lb) and np.array_equal(gub, ub)
