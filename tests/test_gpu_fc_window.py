"""Fully connected layers behind images with known windows (the contraction that stays inside the windows): against the
oracle, with what is left unwritten poisoned, at the edges of its tiles (rows 16 .. 130, columns around multiples of 32 and
64), with windows that are empty, that reach the border and whose union holds more rows than one list.  Every case asserts
that the layer took the path."""
import numpy as np
import pytest

from oracle import nnv_oracle as o
from tests.gpu_util import assert_close, compare_sets
from tests.test_gpu_window_layers import _layers

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _net_layers(rs, names, hw, cin):
    """The layers up to the first FC layer, then FC / ReLU layers on vectors."""
    names = names.split()
    first = next(i for i, nm in enumerate(names) if nm.startswith("fc"))
    layers = _layers(rs, names[:first + 1], hw, cin)
    for nm in names[first + 1:]:
        if nm == "relu":
            layers.append({"type": "relu"})
        else:
            dim = next(L["W"].shape[0] for L in reversed(layers) if L["type"] == "fc")
            layers.append({"type": "fc", "W": rs.randn(int(nm[2:]), dim) / np.sqrt(dim), "b": rs.randn(int(nm[2:])) * 0.1})
    return layers


# hw, channels, layers, sets, half-width of the boxes (wide enough for the unit-vector columns to be worth a gather pass)
NETS = [
    ((16, 16), 1, "conv3_1_1_4 relu conv3_1_1_6 relu fc5 relu fc3", 1, 0.1),
    ((15, 17), 1, "conv3_1_1_4 relu conv3_1_1_9 relu fc32 relu fc3", 1, 0.06),
    ((16, 16), 1, "conv3_1_1_4 relu conv3_1_1_6 relu fc33", 3, 0.02),      # an array
    ((14, 19), 2, "conv3_1_1_5 relu fc64 relu fc20 relu fc2", 1, 0.02),
    ((14, 19), 2, "conv3_1_1_5 relu fc65 relu fc4", 2, 0.02),
    ((16, 16), 1, "conv3_1_1_8 relu conv3_1_1_8 relu fc130 relu fc9", 1, 0.02),  # at least 128 rows: ranges in a kernel of their own
    ((16, 16), 1, "conv3_1_1_6 bn fc96 relu fc6", 1, 0.02),               # no row reset in front of the layer
    ((13, 13), 8, "conv1_2_0_5 fc40 relu fc2", 1, 0.02),                  # three windows of four are empty
    ((50, 44), 1, "conv3_1_1_1 relu fc48 relu fc3", 1, 0.05),             # more window starts than the sort tells apart
    ((12, 12), 1, "conv3_1_1_150 fc70 relu fc5", 2, 0.02),                # thousands of rows per union
    ((28, 28), 1, "conv3_1_1_4 relu conv3_1_1_3 relu fc100 relu fc4", 24, 0.02),  # tiles of 64 columns ...
    ((28, 28), 1, "conv3_1_1_4 relu conv3_1_1_3 relu fc20 relu fc4", 44, 0.02),   # ... and of 32 rows
    ((12, 12), 1, "conv3_1_1_4 relu conv3_1_1_6 relu fc33 relu fc4", 67, 0.05),   # range sums of the other columns by a product
]
COMPARED = 3  # sets of an array that are compared with the oracle: the first ones and the last


@pytest.mark.parametrize("hw,cin,names,count,eps", NETS)
@pytest.mark.parametrize("poison", [False, True])
def test_fc_layer_inside_windows(nnv, hw, cin, names, count, eps, poison):
    rs = np.random.RandomState(len(names) + hw[1])
    layers = _net_layers(rs, names, hw, cin)
    ctx = nnv.default_context()
    bounds = []
    for i in range(count):
        x = rs.rand(*hw, cin)
        e = eps * (rs.rand(*hw, cin) < (0.9 if i else 2.0))
        bounds.append((x - e, x + e))
    dev_in = [nnv.ImageStar(*b) for b in bounds]
    was, before = ctx.switch_is_on("poison_pending"), ctx.routes()["fc_window"]
    ctx.set_switch("poison_pending", poison)
    try:
        net = nnv.NN.from_config(layers)
        net.reach(dev_in if count > 1 else dev_in[0], {"reachMethod": "relax-star-area", "relaxFactor": 1})
        assert ctx.routes()["fc_window"] - before == count, "the first FC layer stays inside the windows"
        at = [li for li, L in enumerate(layers) if L["type"] == "fc"]
        for i in sorted(set(list(range(min(count, COMPARED - 1))) + [count - 1])):
            _, exp = o.nn_reach(layers, o.image_star_from_bounds(*bounds[i]), "relax-star-area", 1.0, keep=True)
            for li in at:
                ds = net.reachSet[li][i] if count > 1 else net.reachSet[li]
                lb, ub = ds.estimateRanges()
                elb, eub = o.image_star_estimate_ranges(exp[li]) if isinstance(exp[li], o.OImageStar) else o.estimate_ranges(exp[li])
                assert_close(lb, elb, "layer %d set %d lb" % (li + 1, i))
                assert_close(ub, eub, "layer %d set %d ub" % (li + 1, i))
                compare_sets(ds, exp[li], "layer %d set %d" % (li + 1, i), check_constraints=False)
    finally:
        ctx.set_switch("poison_pending", was)


@pytest.mark.parametrize("hw,cin,names,eps", [
    ((6, 6), 1, "conv5_1_2_4 relu fc100 relu fc3", 0.05),     # windows as large as the image
    ((16, 16), 1, "conv3_1_1_1 relu fc4 relu fc3", 0.01),     # a product that is bound by its launch
])
def test_fc_layer_over_whole_images(nnv, hw, cin, names, eps):
    rs = np.random.RandomState(7)
    ctx = nnv.default_context()
    net = nnv.NN.from_config(_net_layers(rs, names, hw, cin))
    x = rs.rand(*hw, cin)
    before = ctx.routes()["fc_window"]
    net.reach(nnv.ImageStar(x - eps, x + eps), {"reachMethod": "relax-star-area", "relaxFactor": 1})
    assert ctx.routes()["fc_window"] == before
