"""Infinite bounds, centres and weights through the kernels that leave products with exact zeros out: 0 * Inf is NaN, so
what may be left out with finite numbers may not be with infinite ones, and a sum that does not take part in the reference
(the centre's, in Star.estimateRanges) may not turn into one."""
import numpy as np
import pytest

from oracle import nnv_oracle as o
from tests.gpu_util import assert_close

pytestmark = pytest.mark.gpu

OPTS = {"reachMethod": "relax-star-area", "relaxFactor": 1}


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _same_where_not_finite(got, exp, what):
    got, exp = np.asarray(got), np.asarray(exp)
    assert got.shape == exp.shape, what
    assert np.array_equal(np.isnan(got), np.isnan(exp)), what + ": NaN in other places"
    inf = np.isinf(exp)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], exp[inf]), what + ": other infinities"
    fin = np.isfinite(exp)
    assert_close(got[fin], exp[fin], what)


@pytest.mark.parametrize("channels", [16, 33])
def test_an_infinite_centre_behind_a_convolution_by_position(nnv, channels):
    """An infinite bias makes one channel of the first layer's centre infinite; the second layer's centre is +-Inf all
    over.  Its generators are finite: the bounds are +-Inf, not NaN."""
    rs = np.random.RandomState(channels)
    W1, W2 = rs.randn(3, 3, 1, 16) / 3, rs.randn(3, 3, 16, channels) / 12
    W2[:, :, 3, :] = np.abs(W2[:, :, 3, :]) * np.where(np.arange(channels) % 2 == 0, 1.0, -1.0)
    b1 = rs.randn(16) * 0.1
    b1[3] = np.inf
    conv = lambda W, b: {"type": "conv", "W": W, "b": b, "padding": [1] * 4, "stride": [1, 1], "dilation": [1, 1]}
    layers = [conv(W1, b1), {"type": "relu"}, conv(W2, rs.randn(channels) * 0.1), {"type": "relu"}]
    x = rs.rand(10, 11, 1)
    net = nnv.NN.from_config(layers)
    with np.errstate(invalid="ignore"):
        _, exp = o.nn_reach(layers, o.image_star_from_bounds(x - 0.02, x + 0.02), "relax-star-area", 1.0, keep=True)
        net.reach(nnv.ImageStar(x - 0.02, x + 0.02), OPTS)
        for li in (0, 2):
            lb, ub = net.reachSet[li].estimateRanges()
            elb, eub = o.image_star_estimate_ranges(exp[li])
            assert np.isinf(elb).any() and not np.isnan(elb).any()
            _same_where_not_finite(lb, elb, "layer %d lb" % (li + 1))
            _same_where_not_finite(ub, eub, "layer %d ub" % (li + 1))
        # the step classifies by these bounds: what lies at -Inf is reset, what lies at +Inf is kept
        V = net.reachSet[3].V
        assert not V[np.isneginf(eub)].any() and np.isposinf(V[..., 0][np.isposinf(elb)]).all()


def test_an_infinite_weight_in_an_fc_layer_behind_a_convolution(nnv):
    """Every generator image times an infinite weight: NaN where the image is zero at that weight's row, as in the
    product over whole images."""
    rs = np.random.RandomState(3)
    W1, Wf = rs.randn(3, 3, 1, 6) / 3, rs.randn(33, 16 * 16 * 6) / 40
    Wf[5, 700] = np.inf
    layers = [{"type": "conv", "W": W1, "b": 20.0 + rs.randn(6), "padding": [1] * 4, "stride": [1, 1], "dilation": [1, 1]},
              {"type": "relu"}, {"type": "fc", "W": Wf, "b": rs.randn(33)}]
    x = rs.rand(16, 16, 1)
    net = nnv.NN.from_config(layers)
    with np.errstate(invalid="ignore"):
        _, exp = o.nn_reach(layers, o.image_star_from_bounds(x - 0.02, x + 0.02), "relax-star-area", 1.0, keep=True)
        out = net.reach(nnv.ImageStar(x - 0.02, x + 0.02), OPTS)
        V = exp[2].V.reshape(33, -1)
        assert np.isnan(V[5]).any()
        _same_where_not_finite(np.asarray(out.V).reshape(33, -1), V, "V")


def test_an_infinite_weight_in_a_convolution_by_position(nnv):
    """The same for a convolution whose images have windows: the rows a ReLU step has reset count as zeros inside a
    window, so an infinite weight over them is NaN, whatever way the images are computed."""
    rs = np.random.RandomState(4)
    W1, W2 = rs.randn(3, 3, 1, 16) / 3, rs.randn(3, 3, 16, 32) / 12
    W2[1, 1, 2, 7] = np.inf
    conv = lambda W, b: {"type": "conv", "W": W, "b": b, "padding": [1] * 4, "stride": [1, 1], "dilation": [1, 1]}
    net = nnv.NN.from_config([conv(W1, rs.randn(16) * 0.1), {"type": "relu"}, conv(W2, rs.randn(32) * 0.1), {"type": "relu"}])
    x = rs.rand(12, 12, 1)
    ctx = nnv.default_context()
    got = []
    for eager in (True, False):                     # (with every column in memory the images go by the implicit GEMM)
        ctx.set_eager_columns(eager)
        try:
            net.reach(nnv.ImageStar(x - 0.02, x + 0.02), OPTS)
            out = net.reachSet[2]
            got.append((out.estimateRanges(), np.array(out.V)))
        finally:
            ctx.set_eager_columns(False)
    assert np.isnan(got[0][1]).any()
    _same_where_not_finite(got[1][1], got[0][1], "V")
    _same_where_not_finite(got[1][0][0], got[0][0][0], "lb")
    _same_where_not_finite(got[1][0][1], got[0][0][1], "ub")


@pytest.mark.parametrize("N", [20, 300, 3000])      # one block, several, beyond the one-block classification
@pytest.mark.parametrize("rows", [(4,), (4, 9), ()])
def test_an_infinite_upper_bound_in_front_of_a_relu(nnv, N, rows):
    """A neuron with bounds -Inf .. Inf gets a predicate with upper bound Inf: in Star.estimateRanges of the output every
    other row meets it as 0 * Inf."""
    rs = np.random.RandomState(N + len(rows))
    n = 2
    V = rs.randn(N, n + 1)
    for r in rows:
        V[r] = [0.5, 1.5e308, 1.5e308]              # (finite entries whose sum is not)
    C, d, pl, pu = np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n)
    with np.errstate(invalid="ignore", over="ignore"):
        exp = o.reach_relaxed_star(o.OStar(V, C, d, pl, pu), "relax-star-area")
        elb, eub = o.estimate_ranges(exp)
    out = nnv.ReluLayer().reach(nnv.Star(V, C, d, pl, pu), "relax-star-area", [], 1)
    lb, ub = out.estimateRanges()
    assert np.isnan(elb).all() == (len(rows) > 0)
    _same_where_not_finite(lb, elb, "lb")
    _same_where_not_finite(ub, eub, "ub")
