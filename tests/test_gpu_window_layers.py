"""Row maps and average pooling on generators that are known to be sparse (windows of a convolution, unit vectors of a box
or a ReLU step): against the oracle layer by layer, with what is left unwritten poisoned, in the order written first /
read first, and for the sizes where windows reach the border, overlap or stop paying.  Every case asserts which layers stayed inside windows."""
import numpy as np
import pytest

from oracle import nnv_oracle as o
from tests.gpu_util import assert_close, compare_sets

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _layers(rs, names, hw, cin):
    h, w = hw
    c, out = cin, []
    for nm in names:
        if nm.startswith("conv"):
            k, s, p, co = (int(t) for t in nm[4:].split("_"))
            out.append({"type": "conv", "W": rs.randn(k, k, c, co) / k, "b": rs.randn(co) * 0.1, "padding": [p] * 4, "stride": [s] * 2, "dilation": [1, 1]})
            h, w, c = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1, co
        elif nm == "bn":
            out.append({"type": "batchnorm", "mean": 0.1 * rs.randn(c), "var": rs.rand(c) + 0.5, "eps": 1e-5, "scale": rs.randn(c) * (rs.rand(c) < 0.8),
                        "offset": 0.1 * rs.randn(c)})
        elif nm.startswith("pool"):
            k, s, p = (int(t) for t in nm[4:].split("_"))
            out.append({"type": "avgpool", "pool": [k, k], "stride": [s, s], "padding": [p] * 4})
            h, w = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
        elif nm == "relu":
            out.append({"type": "relu"})
        elif nm == "norm":
            out.append({"type": "imageinput", "normalization": "zscore", "input_size": [h, w, c], "mean": rs.rand(1, 1, c), "std": 0.5 + rs.rand(c)})
        elif nm == "sym":
            out.append({"type": "imageinput", "normalization": "rescale-symmetric", "input_size": [h, w, c], "min": -1.0, "max": 3.0})
        elif nm == "flat":
            out.append({"type": "flatten", "flatten_type": "nnet.keras.layer.FlattenCStyleLayer"})
        else:
            out.append({"type": "fc", "W": rs.randn(int(nm[2:]), h * w * c) / np.sqrt(h * w * c), "b": rs.randn(int(nm[2:])) * 0.1})
    return out


# the last: sets per image that go through a row map in windows, a row map of a box, a pooling in windows
NETS = [
    ((12, 9), 3, "norm conv3_1_1_4 bn relu pool2_2_0 conv3_1_1_5 bn relu pool3_2_1 flat fc7", (1, 1, 1)),
    ((13, 13), 1, "sym bn conv3_1_1_6 bn pool2_2_0 bn relu pool2_1_1 conv3_2_0_4 relu fc5", (2, 2, 2)),
    ((16, 16), 2, "pool2_2_0 bn conv3_1_1_3 relu bn relu fc4", (1, 0, 1)),          # pooling a box; a row map behind a pending reset
    ((17, 16), 1, "norm pool3_2_1 relu pool2_1_1 bn fc6", (1, 1, 2)),
    ((5, 5), 2, "norm conv3_1_1_3 bn relu pool2_2_0 fc3", (1, 1, 0)),                 # windows as large as the image
    ((9, 20), 3, "norm conv5_1_2_3 bn relu pool5_3_2 conv1_1_0_4 relu fc3", (1, 1, 1)),
]


@pytest.mark.parametrize("hw,cin,names,inside", NETS)
@pytest.mark.parametrize("mode", ["default", "poison", "single_dims", "eager", "array"])
def test_sparse_generators_through_row_maps_and_pooling(nnv, hw, cin, names, inside, mode):
    rs = np.random.RandomState(len(names) + hw[0])
    layers = _layers(rs, names.split(), hw, cin)
    count = 3 if mode == "array" else 1
    ctx = nnv.default_context()
    dev_in, ora_in = [], []
    for _ in range(count):
        x = rs.rand(*hw, cin)
        eps = 0.02 * (rs.rand(*hw, cin) < 0.7) if mode == "single_dims" else 0.02
        dev_in.append(nnv.ImageStar(x - eps, x + eps))
        ora_in.append(o.image_star_from_bounds(x - eps, x + eps))
    was = ctx.switch_is_on("poison_pending"), ctx.switch_is_on("eager_cols")
    if mode == "poison":
        ctx.set_switch("poison_pending", True)
    if mode == "eager":
        ctx.set_eager_columns(True)
    try:
        net = nnv.NN.from_config(layers)
        before = ctx.routes()
        out = net.reach(dev_in if count > 1 else dev_in[0], {"reachMethod": "relax-star-area", "relaxFactor": 1})
        took = {k: v - before[k] for k, v in ctx.routes().items()}
        assert (took["rowmap_window"], took["rowmap_box"], took["pool_window"]) == tuple(0 if mode == "eager" else count * k for k in inside), took
        ranges = [(s[0] if count > 1 else s).estimateRanges() for s in net.reachSet[:-1]]   # before any matrix is read
        for i in range(count):
            exp, exp_sets = o.nn_reach(layers, ora_in[i], "relax-star-area", 1.0, keep=True)
            for li, (L, ds, os_) in enumerate(zip(layers, net.reachSet, exp_sets)):
                tag = "layer %d (%s) set %d" % (li + 1, L["type"], i)
                ds = ds[i] if count > 1 else ds
                if i == 0 and li < len(layers) - 1:
                    elb, eub = o.image_star_estimate_ranges(os_) if isinstance(os_, o.OImageStar) else o.estimate_ranges(os_)
                    assert_close(ranges[li][0], elb, tag + " lb")
                    assert_close(ranges[li][1], eub, tag + " ub")
                compare_sets(ds, os_, tag, check_constraints=False)
            compare_sets(out[i] if count > 1 else out, exp, "output", check_constraints=True)
    finally:
        ctx.set_switch("poison_pending", was[0])
        ctx.set_eager_columns(was[1])


def test_an_array_goes_in_one_launch_per_layer(nnv):
    """Twenty images with different numbers of predicates, one of them listed twice: one launch per row map and pooling, the
    same sets to the bit as every image gives by itself."""
    rs = np.random.RandomState(5)
    hw, cin, names = (12, 11), 3, "norm conv3_1_1_4 bn relu pool2_2_0 pool2_1_0 relu".split()
    layers = _layers(rs, names, hw, cin)
    ctx = nnv.default_context()
    net = nnv.NN.from_config(layers)
    opts = {"reachMethod": "relax-star-area", "relaxFactor": 1}
    bounds = []
    for i in range(20):
        x, eps = rs.rand(*hw, cin), 0.02 * (rs.rand(*hw, cin) < 0.2 + 0.04 * i)
        bounds.append((x - eps, x + eps))
    sets = [nnv.ImageStar(*b) for b in bounds]
    before = ctx.routes()
    ctx.set_timing(2)
    try:
        ctx.kernel_time(4)
        net.reach(sets + [sets[3]], opts)
        _, launches, _ = ctx.kernel_time(4)
    finally:
        ctx.set_timing(0)
    took = {k: v - before[k] for k, v in ctx.routes().items()}
    assert (took["rowmap_box"], took["rowmap_window"], took["pool_window"]) == (21, 21, 42), took
    assert launches == 4, "one launch per row map and pooling layer"
    got = [[(s.estimateRanges(), np.array(s.V)) for s in layer] for layer in net.reachSet]
    for i, b in list(enumerate(bounds)) + [(20, bounds[3])]:
        net.reach(nnv.ImageStar(*b), opts)
        for li, out in enumerate(net.reachSet):
            (lb, ub), V = got[li][i]
            assert np.array_equal(V, np.array(out.V)), (li, i)
            elb, eub = out.estimateRanges()
            assert_close(lb, elb, "lb")
            assert_close(ub, eub, "ub")
