"""The kernels that place crossing neurons by counting the entries in front of them, at their edges: 16 entries to a block and 64 rows to
a wave in the kernel for a few sets of at most 2048 neurons; in the one for larger sets (and for lists of more than 1024 of many sets at
once) blocks of 32 entries, steps of 128 keys, two to a load, and pieces of 4096 keys in LDS.  Classes, order (ties by neuron index)
and the bounds of the new predicates are whole numbers and copies: exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _bounds(rs, N, share):
    """Half-widths and centres are small multiples of 1/8, so that the estimated ranges are exact and many keys tie."""
    half = rs.randint(1, 9, N) / 8.0
    centre = np.where(rs.rand(N) < share, 0.0, np.where(rs.rand(N) < 0.5, 2.0, -2.0)) + rs.randint(0, 2, N) / 16.0
    return centre - half, centre + half


def _bounds_crossing(rs, N, m):
    """The same with exactly m neurons that cross, anywhere."""
    half = rs.randint(1, 9, N) / 8.0
    centre = np.where(rs.rand(N) < 0.5, 2.0, -2.0)
    centre[rs.permutation(N)[:m]] = 0.0
    centre += rs.randint(0, 2, N) / 16.0
    return centre - half, centre + half


def _expected(lb, ub, method):
    cross = np.flatnonzero((lb < 0) & (ub > 0))
    key = {"relax-star-area": 0.5 * (np.abs(ub) * np.abs(lb)), "relax-star-range": ub - lb}.get(method)
    return int(np.sum(ub <= 0)), cross if key is None else cross[np.argsort(-key[cross], kind="stable")]


# sets, neurons, share that crosses; above 2048 neurons the classification has two passes of several blocks and the ranking is a launch of its own
CASES = [(c, n, 0.9) for c in (1, 2, 25, 128, 129) for n in (1, 15, 16, 17, 63, 65, 130)]
CASES += [(1, 1023, 1.0), (1, 1025, 1.0), (1, 2047, 1.0), (1, 2048, 0.5), (9, 1024, 1.0), (128, 1040, 0.7), (129, 1040, 1.0), (128, 2048, 0.3), (3, 500, 0.0)]
CASES += [(1, 2049, 0.02), (1, 2050, 1.0), (1, 4097, 0.97), (3, 2111, 0.5), (40, 2300, 1.0), (2, 9000, 0.9), (1, 2100, 0.0)]


@pytest.mark.parametrize("method", ["relax-star-area", "relax-star-range"])
@pytest.mark.parametrize("count,N,share", CASES)
def test_order_of_crossing_neurons(nnv, count, N, share, method):
    rs = np.random.RandomState(N + count)
    _check_order(nnv, *(np.stack(x, axis=1) for x in zip(*[_bounds(rs, N, share) for _ in range(count)])), method)


# list lengths around a block's entries (multiples of 32), a step's keys (128) and a piece (4096)
@pytest.mark.parametrize("method", ["relax-star-area", "relax-star-range"])
@pytest.mark.parametrize("m", [1, 31, 32, 33, 127, 128, 129, 2079, 2080, 2081, 2175, 2176, 2177, 4063, 4064, 4065, 4095, 4096, 4097, 4127, 4128, 4129, 4225])
@pytest.mark.parametrize("count,N", [(1, 5000), (3, 4400)])
def test_lengths_of_long_lists(nnv, count, N, m, method):
    rs = np.random.RandomState(N + m)
    lb, ub = (np.stack(x, axis=1) for x in zip(*[_bounds_crossing(rs, N, m + i) for i in range(count)]))
    assert np.sum((lb[:, 0] < 0) & (ub[:, 0] > 0)) == m
    _check_order(nnv, lb, ub, method)


def _check_order(nnv, lb, ub, method):
    N, count = lb.shape
    sets = nnv.Star.from_boxes(lb, ub) if count > 1 else nnv.Star(lb[:, 0], ub[:, 0])
    out = nnv.layers.ReluLayer().reach(sets, method, [], 1, None, "linprog")
    for i in sorted({0, count // 2, count - 1}):
        o = out[i] if count > 1 else out
        inactive, order = _expected(lb[:, i], ub[:, i], method)
        ni, idx, clb, cub = o.relu_info()
        assert ni == inactive and np.array_equal(idx, order), "set %d" % i
        assert np.array_equal(clb, lb[order, i]) and np.array_equal(cub, ub[order, i])
        assert np.array_equal(o.predicate_lb[N:], np.zeros(order.size)) and np.array_equal(o.predicate_ub[N:], ub[order, i])
        # the rows that pass, as the layer behind sees them: centre, generators of the set before, unit vectors behind
        if N <= 130:
            V = np.array(o.V)
            kept = (ub[:, i] > 0) & ~((lb[:, i] < 0) & (ub[:, i] > 0))
            assert np.array_equal(V[:, 0], np.where(kept, 0.5 * (lb[:, i] + ub[:, i]), 0.0))
            assert np.array_equal(V[:, 1:N + 1], np.diag(np.where(kept, 0.5 * (ub[:, i] - lb[:, i]), 0.0)))
            assert np.array_equal(V[:, N + 1:], np.eye(N)[:, order])
