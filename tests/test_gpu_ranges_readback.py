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


@pytest.mark.parametrize("N,count", [(1, 1), (1, 3), (2, 2), (15, 1), (16, 3), (17, 20), (127, 2), (130, 1)])
@pytest.mark.parametrize("all_wide", [True, False])
def test_a_box_is_written_when_its_matrix_is_read(N, count, all_wide):
    """Star(lb, ub) keeps its centre and a list of scaled unit vectors; V, the ranges (pooled and without allocation), a
    ReLU step and the first layer's map see the matrix of the reference all the same.  Half-widths are mixed in sign
    (ub < lb is allowed) and partly zero."""
    import nnv_amd as nnv
    from nnv_amd import _lib
    from oracle import nnv_oracle as oracle
    from tests.gpu_util import DeviceDoubles, assert_close
    rs = np.random.RandomState(7 * N + count)
    lbs = rs.randn(N, count)
    ubs = lbs + rs.rand(N, count) * (1.0 if all_wide else (rs.rand(N, count) < 0.6)) * (1.0 if all_wide else np.where(rs.rand(N, count) < 0.2, -1.0, 1.0))
    exp = [oracle.star_from_box(lbs[:, i], ubs[:, i]) for i in range(count)]
    ctx = nnv.default_context()
    sets = nnv.Star.from_boxes(lbs, ubs)
    buf = DeviceDoubles(N)
    for i in range(count):
        _lib.check(ctx.lib.nnvhip_estimate_ranges_static(ctx.handle, sets[i]._h.h, buf.ptr, None))
        ctx.synchronize()
        assert np.array_equal(buf.get(), oracle.estimate_ranges(exp[i])[0])
    lb, ub = nnv.Star.estimateRanges_array(sets)
    for i in range(count):
        assert np.array_equal(lb[:, i], oracle.estimate_ranges(exp[i])[0]) and np.array_equal(ub[:, i], oracle.estimate_ranges(exp[i])[1])
        assert sets[i].nVar == exp[i].V.shape[1] - 1
    fresh = nnv.Star.from_boxes(lbs, ubs)
    relu = nnv.ReluLayer().reach(fresh, "relax-star-area", [], 1)
    relu = relu if count > 1 or isinstance(relu, (list, nnv.SetArray)) else [relu]
    W, b = rs.randn(33, N), rs.randn(33)
    mapped = nnv.FullyConnectedLayer(W, b).reach(nnv.Star.from_boxes(lbs, ubs), "relax-star-area")
    for i in range(count):
        assert np.array_equal(sets[i].V, exp[i].V) and np.array_equal(fresh[i].V, exp[i].V)
        assert_close(mapped[i].V, oracle.affine_map(exp[i], W, b).V, "W * box")
        assert np.array_equal(relu[i].V, oracle.reach_relaxed_star(exp[i], "relax-star-area").V)


@pytest.mark.parametrize("N,count", [(1, 1), (255, 1), (257, 3), (2500, 1)])
@pytest.mark.parametrize("eager", [False, True])
def test_ranges_of_a_relu_output_come_from_its_input(N, count, eager):
    """Ranges of a ReLU step's output without its matrix: against the scan of that matrix by the oracle, with the matrix
    written by the step or not, one-block and multi-block classification."""
    import nnv_amd as nnv
    from oracle import nnv_oracle as oracle
    from tests.gpu_util import assert_close_elementwise
    rs = np.random.RandomState(N + count)
    ctx = nnv.default_context()
    n = 9
    sets, exp = [], []
    for _ in range(count):
        V = rs.randn(N, n + 1)
        V[rs.rand(N) < 0.1] = 0.0                    # rows with lb = ub = 0
        V[:, 1:] *= 0.3
        C, d, pl, pu = np.zeros((1, n)), np.zeros(1), -rs.rand(n), rs.rand(n)
        sets.append(nnv.Star(V, C, d, pl, pu))
        exp.append(oracle.reach_relaxed_star(oracle.OStar(V, C, d, pl, pu), "relax-star-area"))
    ctx.set_eager_relu(eager)
    try:
        out = nnv.ReluLayer().reach(sets, "relax-star-area", [], 1)
    finally:
        ctx.set_eager_relu(False)
    lb, ub = nnv.Star.estimateRanges_array(out)
    for i in range(count):
        ol, ou = oracle.estimate_ranges(exp[i])
        assert_close_elementwise(lb[:, i], ol, "lb")
        assert_close_elementwise(ub[:, i], ou, "ub")
        assert np.array_equal(out[i].V, exp[i].V)
