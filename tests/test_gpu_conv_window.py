"""Convolutions that go by output position (images with windows): against the oracle, with what is left unwritten poisoned, at
the edges of the channel tiles (16, 32, 64), with more columns per position than one list holds and more than one part,
with strides, dilation, borders, empty windows and without a kept row; in an array and by itself (to the bit, without dilation).  Every case asserts which
layers went by position."""
import numpy as np
import pytest

from oracle import nnv_oracle as o
from tests.gpu_util import assert_close, compare_sets

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _layers(rs, hw, cin, convs, bias):
    out, c, (h, w) = [], cin, hw
    for k, s, p, d, co in convs:
        b = rs.randn(co) * 0.1 + (bias if len(out) == 0 else 0.0)
        out.append({"type": "conv", "W": rs.randn(k, k, c, co) / k, "b": b, "padding": [p] * 4, "stride": [s] * 2, "dilation": [d] * 2})
        out.append({"type": "relu"})
        h, w, c = (h + 2 * p - d * (k - 1) - 1) // s + 1, (w + 2 * p - d * (k - 1) - 1) // s + 1, co
    return out


# (filter, stride, padding, dilation, channels) per layer; bias of the first layer: -20 leaves no row, +20 every row; how many
# layers go by position; whether a position's columns come in several parts there
NETS = [
    ((9, 11), 1, [(3, 1, 1, 1, 16), (3, 1, 1, 1, 16)], 0.0, 1, False),
    ((9, 11), 1, [(3, 1, 1, 1, 14), (3, 2, 1, 1, 17)], 0.0, 1, False),
    ((12, 10), 1, [(3, 1, 1, 1, 8), (3, 1, 1, 1, 33), (3, 2, 0, 1, 64)], 0.0, 1, False),
    ((10, 10), 2, [(3, 1, 1, 1, 6), (3, 1, 1, 1, 65)], 0.0, 1, False),
    ((24, 26), 3, [(5, 2, 2, 1, 16), (3, 1, 1, 1, 32), (3, 1, 0, 1, 20)], 0.0, 2, True),
    ((14, 12), 1, [(3, 1, 1, 1, 16), (3, 1, 2, 2, 32)], 0.0, 1, False),
    ((11, 11), 1, [(1, 2, 0, 1, 40), (1, 1, 0, 1, 60)], 0.0, 1, False),
    ((8, 8), 40, [(1, 1, 0, 1, 20), (3, 1, 1, 1, 16)], 0.0, 1, True),      # 360 columns per position
    ((9, 9), 1, [(3, 1, 1, 1, 16), (3, 1, 1, 1, 16)], -20.0, 1, False),
    ((9, 9), 1, [(3, 1, 1, 1, 16), (3, 1, 1, 1, 16)], 20.0, 1, False),
]


@pytest.mark.parametrize("hw,cin,convs,bias,by_position,parts", NETS)
@pytest.mark.parametrize("poison", [False, True])
def test_convolution_by_position(nnv, hw, cin, convs, bias, by_position, parts, poison):
    rs = np.random.RandomState(hw[0] + 31 * cin + len(convs))
    layers = _layers(rs, hw, cin, convs, bias)
    opts = {"reachMethod": "relax-star-area", "relaxFactor": 1}
    boxes = []
    for i in range(2):
        x = rs.rand(*hw, cin)
        eps = 0.02 * (rs.rand(*hw, cin) < (0.8 if i else 2.0))
        boxes.append((x - eps, x + eps))
    ctx = nnv.default_context()
    was = ctx.switch_is_on("poison_pending")
    ctx.set_switch("poison_pending", poison)
    try:
        net = nnv.NN.from_config(layers)
        before = ctx.routes()
        net.reach([nnv.ImageStar(*b) for b in boxes], opts)
        took = {k: v - before[k] for k, v in ctx.routes().items()}
        assert took["conv_window"] == 2 * by_position and (took["conv_window_parts"] > 0) == parts, took
        arr = [[(s.estimateRanges(), np.array(s.V)) for s in layer] for layer in net.reachSet]
        for i, b in enumerate(boxes):
            net.reach(nnv.ImageStar(*b), opts)
            _, exp = o.nn_reach(layers, o.image_star_from_bounds(*b), "relax-star-area", 1.0, keep=True)
            for li, (ds, es) in enumerate(zip(net.reachSet, exp)):
                tag = "layer %d set %d" % (li + 1, i)
                lb, ub = ds.estimateRanges()
                elb, eub = o.image_star_estimate_ranges(es)
                assert_close(lb, elb, tag + " lb")
                assert_close(ub, eub, tag + " ub")
                compare_sets(ds, es, tag, check_constraints=False)
                (alb, aub), aV = arr[li][i]
                assert np.array_equal(np.array(ds.V), aV), tag
                if all(d == 1 for _, _, _, d, _ in convs):
                    assert np.array_equal(lb, alb) and np.array_equal(ub, aub), tag
                else:  # (the stamps of a dilated filter are summed in a pass that cuts by the size of the call)
                    assert_close(alb, elb, tag + " array lb")
                    assert_close(aub, eub, tag + " array ub")
    finally:
        ctx.set_switch("poison_pending", was)
