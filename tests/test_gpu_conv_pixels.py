"""Convolution outputs kept pixel by pixel between two layers of one reach call: against the oracle and against the same layers called
one by one (which write columns), with what is left unwritten poisoned; at the edges of channel tiles, windows that wrap around their
bound, borders, strides, empty windows, one set and arrays.  And every other reader of such a set: its columns, a pooling, a row
map, an FC layer without windows, a convolution that does not go by position.  Every case asserts which layers kept pixels.
Tolerance: the products are the same, their sums of up to K = 1100 terms are added in another order, |difference| <= 2 K eps of the
largest sum of magnitudes, which for these nets stays below 50 times the largest value: 2.5e-11."""
import numpy as np
import pytest

from oracle import nnv_oracle as o
from tests.gpu_util import assert_close, compare_sets, flat_V

pytestmark = pytest.mark.gpu
TOL = 2.5e-11


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _layers(rs, hw, cin, convs, fc):
    out, c, (h, w) = [], cin, hw
    for k, s, p, co in convs:
        out.append({"type": "conv", "W": rs.randn(k, k, c, co) / k, "b": rs.randn(co) * 0.1, "padding": [p] * 4, "stride": [s] * 2, "dilation": [1, 1]})
        out.append({"type": "relu"})
        h, w, c = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1, co
    if fc:
        out.append({"type": "fc", "W": rs.randn(fc, h * w * c) / np.sqrt(h * w * c), "b": rs.randn(fc)})
    return out


# image, channels, (filter, stride, padding, channels) per layer, rows of an FC layer at the end (0: none), layers that keep pixels
NETS = [
    ((12, 11), 1, [(3, 1, 1, 16), (3, 1, 1, 16)], 0, 1),
    ((13, 9), 2, [(3, 1, 0, 15), (3, 2, 1, 17), (3, 1, 1, 33)], 0, 1),
    ((20, 22), 1, [(3, 1, 1, 17), (3, 1, 1, 40), (3, 2, 0, 64)], 70, 3),
    ((24, 20), 3, [(5, 2, 2, 16), (3, 1, 1, 65)], 24, 2),
    ((11, 11), 1, [(1, 2, 0, 40), (1, 1, 0, 60)], 100, 2),
    ((17, 16), 1, [(3, 1, 1, 8), (3, 1, 1, 16)], 90, 0),         # the second convolution is too small to go by position
]


def _boxes(rs, hw, cin, count):
    out = []
    for i in range(count):
        x = rs.rand(*hw, cin)
        eps = 0.01 * (rs.rand(*hw, cin) < (2.0, 0.7, 0.05)[i % 3])
        out.append((x - eps, x + eps))
    return out


def _one_by_one(nnv, net, sets):
    out = []
    for L in net.Layers:
        sets = L.reach(sets, "relax-star-area", [], 1, None, "linprog")
        out.append(sets)
    return out


@pytest.mark.parametrize("hw,cin,convs,fc,kept", NETS)
@pytest.mark.parametrize("count", [1, 3])
def test_pixels_between_layers(nnv, hw, cin, convs, fc, kept, count):
    rs = np.random.RandomState(hw[0] + 31 * cin + len(convs))
    layers = _layers(rs, hw, cin, convs, fc)
    boxes = _boxes(rs, hw, cin, count)
    ctx = nnv.default_context()
    was = ctx.switch_is_on("poison_pending")
    ctx.set_switch("poison_pending", True)
    try:
        net = nnv.NN.from_config(layers)
        sets = [nnv.ImageStar(*b) for b in boxes]
        before = ctx.routes()
        net.reach(sets if count > 1 else sets[0], {"reachMethod": "relax-star-area", "relaxFactor": 1})
        took = ctx.routes()["conv_pixels"] - before["conv_pixels"]
        assert took == kept * count
        plain = _one_by_one(nnv, net, [nnv.ImageStar(*b) for b in boxes] if count > 1 else nnv.ImageStar(*boxes[0]))
        assert ctx.routes()["conv_pixels"] - before["conv_pixels"] == took       # (nothing was known about the layers behind)
        for i in range(count):
            _, exp = o.nn_reach(layers, o.image_star_from_bounds(*boxes[i]), "relax-star-area", 1.0, keep=True)
            for li, es in enumerate(exp):
                ds, ps = (net.reachSet[li][i], plain[li][i]) if count > 1 else (net.reachSet[li], plain[li])
                tag = "layer %d set %d" % (li + 1, i)
                lb, ub = ds.estimateRanges()
                plb, pub = ps.estimateRanges()
                assert_close(lb, plb, tag + " lb", TOL)
                assert_close(ub, pub, tag + " ub", TOL)
                assert_close(np.array(ds.V), np.array(ps.V), tag + " V", TOL)
                compare_sets(ds, es, tag, check_constraints=layers[li]["type"] == "relu")
    finally:
        ctx.set_switch("poison_pending", was)


def test_other_readers_of_kept_pixels(nnv):
    rs = np.random.RandomState(5)
    hw, cin = (18, 16), 1
    layers = _layers(rs, hw, cin, [(3, 1, 1, 16), (3, 1, 1, 32)], 40)
    net = nnv.NN.from_config(layers)
    (lb, ub), = _boxes(rs, hw, cin, 1)
    readers = [nnv.layers.Conv2DLayer(rs.randn(3, 3, 16, 4), rs.randn(4), [1] * 4, [2, 2], [1, 1]),
               nnv.layers_affine.AveragePooling2DLayer([2, 2], [2, 2], [0] * 4),
               nnv.layers_affine.BatchNormalizationLayer(NumChannels=16, TrainedMean=rs.rand(16), TrainedVariance=rs.rand(16) + 0.5, Epsilon=1e-5,
                                                         Scale=rs.rand(16), Offset=rs.randn(16)),
               nnv.layers.FullyConnectedLayer(rs.randn(3, 16 * hw[0] * hw[1]), rs.randn(3)), nnv.layers.ReluLayer()]
    ctx = nnv.default_context()
    was = ctx.switch_is_on("poison_pending")
    ctx.set_switch("poison_pending", True)
    try:
        plain = _one_by_one(nnv, net, nnv.ImageStar(lb, ub))
        for at in (0, 1):                                    # the convolution's output, the ReLU step's (its rows not yet reset)
            for L in readers:
                before = ctx.routes()["conv_pixels"]
                net.reach(nnv.ImageStar(lb, ub), {"reachMethod": "relax-star-area", "relaxFactor": 1})
                assert ctx.routes()["conv_pixels"] > before
                got = L.reach(net.reachSet[at], "relax-star-area", [], 1, None, "linprog")
                exp = L.reach(plain[at], "relax-star-area", [], 1, None, "linprog")
                tag = "%s on layer %d" % (type(L).__name__, at + 1)
                assert_close(np.array(got.V), np.array(exp.V), tag, TOL)
                for a, b in zip(got.estimateRanges(), exp.estimateRanges()):
                    assert_close(a, b, tag, TOL)
                assert_close(np.array(net.reachSet[at].V), np.array(plain[at].V), tag + ": its input", TOL)
    finally:
        ctx.set_switch("poison_pending", was)


@pytest.mark.parametrize("count", [1, 3])
@pytest.mark.parametrize("convs,kept", [([(3, 1, 1, 16), (3, 1, 1, 40)], 0), ([(3, 1, 1, 17), (3, 1, 1, 40), (3, 2, 0, 64)], 1)])
def test_a_convolution_at_the_end_reads_columns(nnv, convs, kept, count):
    """The layer that hands the result back writes every column, which the kernel that reads pixels does not do."""
    rs = np.random.RandomState(len(convs))
    hw, cin = (20, 22), 1
    layers = _layers(rs, hw, cin, convs, 0)[:-1]
    boxes = _boxes(rs, hw, cin, count)
    ctx = nnv.default_context()
    net = nnv.NN.from_config(layers)
    sets = [nnv.ImageStar(*b) for b in boxes]
    before = ctx.routes()
    out = net.reach(sets if count > 1 else sets[0], {"reachMethod": "relax-star-area", "relaxFactor": 1})
    assert ctx.routes()["conv_pixels"] - before["conv_pixels"] == kept * count
    for i in range(count):
        exp = o.nn_reach(layers, o.image_star_from_bounds(*boxes[i]), "relax-star-area", 1.0)
        compare_sets(out[i] if count > 1 else out, exp, "set %d" % i)


def test_an_fc_layer_that_reads_columns(nnv):
    """An FC layer stays inside the windows of all sets of an array, or of none: not where a weight is infinite (0 * Inf is NaN), and not
    where the windows of one set are others, as those of an image without generators."""
    rs = np.random.RandomState(3)
    hw, cin = (20, 22), 1
    layers = _layers(rs, hw, cin, [(3, 1, 1, 16)], 70)
    (box, _, _), point = _boxes(rs, hw, cin, 3), rs.rand(*hw, cin)
    wild = [dict(L) for L in layers]
    wild[-1]["W"] = layers[-1]["W"].copy()
    wild[-1]["W"][3, 5] = np.inf
    ctx = nnv.default_context()
    for net, bounds, kept in ((layers, [box], 1), (layers, [box, box], 2), (layers, [box, (point, point)], 0), (wild, [box], 0)):
        sets = [nnv.ImageStar(*b) for b in bounds]
        before = ctx.routes()["conv_pixels"]
        n = nnv.NN.from_config(net)
        out = n.reach(sets if len(sets) > 1 else sets[0], {"reachMethod": "relax-star-area", "relaxFactor": 1})
        assert ctx.routes()["conv_pixels"] - before == kept
        plain = _one_by_one(nnv, n, [nnv.ImageStar(*b) for b in bounds] if len(sets) > 1 else nnv.ImageStar(*bounds[0]))[-1]
        for i in range(len(sets)):
            got, exp = (flat_V(x[i] if len(sets) > 1 else x) for x in (out, plain))
            rows = np.arange(70) != 3 if net is wild else slice(None)
            assert_close(got[rows], exp[rows], "set %d" % i, TOL)
            assert np.array_equal(np.isfinite(got), np.isfinite(exp))


def test_without_room_for_pixels(nnv):
    """Memory in which a reach fits with columns is enough: pixels come on top of the matrices, and are done without."""
    rs = np.random.RandomState(8)
    hw, cin = (20, 22), 1
    layers = _layers(rs, hw, cin, [(3, 1, 1, 17), (3, 1, 1, 40), (3, 2, 0, 64)], 70)
    ctx = nnv.default_context()
    net = nnv.NN.from_config(layers)
    (lb, ub), = _boxes(rs, hw, cin, 1)
    options = {"reachMethod": "relax-star-area", "relaxFactor": 1}

    def reach():
        out = net.reach(nnv.ImageStar(lb, ub), options)
        return [np.array(x) for x in out.estimateRanges()]

    def nothing_cached():
        net.reachSet = []
        ctx.synchronize()
        ctx.trim_pool()

    was = ctx.switch_is_on("no_conv_pixels")
    before = ctx.routes()["conv_pixels"]
    ctx.set_switch("no_conv_pixels", True)
    try:
        reach()                                              # (the weights are on the device from here on)
        nothing_cached()
        exp = reach()
        room = sum(ctx.pool_stats())
        assert ctx.routes()["conv_pixels"] == before
        ctx.set_switch("no_conv_pixels", False)
        nothing_cached()
        reach()
        took = ctx.routes()["conv_pixels"] - before
        assert took > 0 and sum(ctx.pool_stats()) > room     # it does come on top
        for some in (room, room + (sum(ctx.pool_stats()) - room) // 2):
            ctx.debug_pool_limit(some)
            for _ in range(2):
                nothing_cached()
                for a, b in zip(reach(), exp):
                    assert_close(a, b, "room for %d bytes" % some, TOL)
                assert sum(ctx.pool_stats()) <= some
            ctx.debug_pool_limit(0)
    finally:
        ctx.debug_pool_limit(0)
        ctx.set_switch("no_conv_pixels", was)
