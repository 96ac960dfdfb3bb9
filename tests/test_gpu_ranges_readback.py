"""estimateRanges on the host: the read-back for every size of result, from one value to past the limit at which the
copy engine takes over (4096 values per block of the posting kernel, 2^17 values in all)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,count", [(1, 1), (7, 1), (2048, 1), (2049, 1), (10, 1), (10, 205), (17, 130), (512, 128), (512, 129), (70000, 1)])
def test_ranges_of_boxes_come_back_whole(N, count):
    from nnv_amd import Star
    rs = np.random.RandomState(N + count)
    lbs = rs.randn(N, count)
    ubs = lbs + rs.rand(N, count) * (rs.rand(N, count) < (0.9 if N < 5000 else 0.01))  # (some dimensions without width)
    sets = Star.from_boxes(lbs, ubs)
    lb, ub = Star.estimateRanges_array(sets)
    c, v = 0.5 * (lbs + ubs), 0.5 * (ubs - lbs)
    # one generator per row: the sums are single products with -1 / +1, so the values are exact
    assert np.array_equal(lb, c - v) and np.array_equal(ub, c + v)
    again = Star.estimateRanges_array(sets)
    assert np.array_equal(again[0], lb) and np.array_equal(again[1], ub)
    one = sets[count - 1].estimateRanges()
    assert np.array_equal(one[0], lb[:, -1]) and np.array_equal(one[1], ub[:, -1])
