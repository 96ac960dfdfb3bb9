"""Fully connected layers behind images with known windows (the contraction that stays inside the windows): against the
oracle, with what is left unwritten poisoned, at the edges of its tiles (rows 16 .. 130, columns around multiples of 32 and
64), with windows that are empty, that reach the border and whose union holds more rows than one list."""
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


NETS = [
    ((16, 16), 1, "conv3_1_1_4 relu conv3_1_1_6 relu fc5 relu fc3", 1),
    ((15, 17), 1, "conv3_1_1_4 relu conv3_2_1_9 relu fc32 relu fc3", 1),
    ((16, 16), 1, "conv3_1_1_4 relu conv3_1_1_6 relu fc33", 3),            # an array
    ((14, 19), 2, "conv3_1_1_5 relu fc64 relu fc20 relu fc2", 1),
    ((14, 19), 2, "conv3_1_1_5 relu fc65 relu fc4", 2),
    ((16, 16), 3, "conv5_2_2_12 relu conv3_1_1_8 relu fc130 relu fc9", 1),   # at least 128 rows: ranges in a kernel of their own
    ((16, 16), 1, "conv3_1_1_6 bn fc96 relu fc6", 1),                      # no row reset in front of the layer
    ((13, 13), 8, "conv1_2_0_5 fc40 relu fc2", 1),                         # three windows of four are empty
    ((50, 44), 1, "conv3_1_1_1 relu fc48", 1),                             # more window starts than the sort tells apart
    ((12, 12), 1, "conv3_1_1_150 fc70 relu fc5", 2),                       # thousands of rows per union
    ((16, 16), 1, "conv3_1_1_16 relu conv3_1_1_6 relu fc100", 20),         # tiles of 64 columns
]


@pytest.mark.parametrize("hw,cin,names,count", NETS)
@pytest.mark.parametrize("poison", [False, True])
def test_fc_layer_inside_windows(nnv, hw, cin, names, count, poison):
    rs = np.random.RandomState(len(names) + hw[1])
    layers = _net_layers(rs, names, hw, cin)
    ctx = nnv.default_context()
    dev_in, ora_in = [], []
    for i in range(count):
        x = rs.rand(*hw, cin)
        eps = 0.01 * (i + 1) * (rs.rand(*hw, cin) < (0.9 if i else 2.0))
        dev_in.append(nnv.ImageStar(x - eps, x + eps))
        ora_in.append(o.image_star_from_bounds(x - eps, x + eps))
    was = ctx.switch_is_on("poison_pending")
    ctx.set_switch("poison_pending", poison)
    try:
        net = nnv.NN.from_config(layers)
        net.reach(dev_in if count > 1 else dev_in[0], {"reachMethod": "relax-star-area", "relaxFactor": 1})
        at = [li for li, L in enumerate(layers) if L["type"] == "fc"]
        for i in range(min(count, 3)):
            _, exp = o.nn_reach(layers, ora_in[i], "relax-star-area", 1.0, keep=True)
            for li in at:
                ds = net.reachSet[li][i] if count > 1 else net.reachSet[li]
                lb, ub = ds.estimateRanges()
                elb, eub = o.image_star_estimate_ranges(exp[li]) if isinstance(exp[li], o.OImageStar) else o.estimate_ranges(exp[li])
                assert_close(lb, elb, "layer %d set %d lb" % (li + 1, i))
                assert_close(ub, eub, "layer %d set %d ub" % (li + 1, i))
                compare_sets(ds, exp[li], "layer %d set %d" % (li + 1, i), check_constraints=False)
    finally:
        ctx.set_switch("poison_pending", was)
