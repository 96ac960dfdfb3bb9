"""Convolutions of an array of image sets in one launch: every set comes out as it does by itself, to the bit, whatever the
others in the array look like (boxes with and without widths, images with dense generators, sets a ReLU left without a
crossing neuron, one handle listed twice), with what is left unwritten poisoned as well."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _net(nnv, rs, hw, cin, convs):
    layers, c, (h, w) = [], cin, hw
    for k, s, p, d, co in convs:
        layers.append({"type": "conv", "W": rs.randn(k, k, c, co) / k, "b": rs.randn(co) * 0.1, "padding": [p] * 4, "stride": [s] * 2, "dilation": [d] * 2})
        layers.append({"type": "relu"})
        h, w, c = (h + 2 * p - d * (k - 1) - 1) // s + 1, (w + 2 * p - d * (k - 1) - 1) // s + 1, co
    layers.append({"type": "fc", "W": rs.randn(5, h * w * c) / np.sqrt(h * w * c), "b": rs.randn(5)})
    return nnv.NN.from_config(layers)


def _sets(nnv, rs, hw, cin):
    def box(eps):
        x = rs.rand(*hw, cin)
        return nnv.ImageStar(x - eps, x + eps)

    some = 0.05 * (rs.rand(*hw, cin) < 0.3)
    V = np.concatenate([rs.rand(*hw, cin, 1), 0.05 * rs.randn(*hw, cin, 4)], axis=3)
    dense = nnv.ImageStar(V, np.zeros((1, 4)), np.zeros((1, 1)), -np.ones(4), np.ones(4))
    return [box(0.02), box(0.0), dense, box(some), box(1e-9), box(0.3)]


# the last two: more than 4096 input rows (two blocks build the pixel table), a dilated filter (stamps in a pass of their own)
@pytest.mark.parametrize("hw,cin,convs", [
    ((9, 7), 1, [(3, 1, 1, 1, 3), (3, 2, 0, 1, 17)]),
    ((16, 16), 3, [(3, 1, 1, 1, 8), (3, 2, 1, 1, 16), (3, 1, 1, 1, 4)]),
    ((14, 14), 2, [(5, 2, 2, 1, 33), (1, 1, 0, 1, 6)]),
    ((40, 37), 3, [(3, 2, 1, 1, 4), (3, 2, 0, 1, 5)]),
    ((15, 12), 1, [(3, 1, 0, 2, 4), (3, 1, 1, 1, 5)]),
])
@pytest.mark.parametrize("poison", [False, True])
def test_array_equals_its_sets_one_by_one(nnv, hw, cin, convs, poison):
    rs = np.random.RandomState(hw[0] * 7 + cin)
    ctx = nnv.default_context()
    net = _net(nnv, rs, hw, cin, convs)
    opts = {"reachMethod": "relax-star-area", "relaxFactor": 1}
    state = rs.get_state()
    sets = _sets(nnv, rs, hw, cin)
    was = ctx.switch_is_on("poison_pending")
    ctx.set_switch("poison_pending", poison)
    try:
        net.reach(sets + [sets[3]], opts)
        got = [[(s.estimateRanges(), np.array(s.V)) for s in layer] for layer in net.reachSet]
        assert all(np.array_equal(layer[3][1], layer[6][1]) for layer in got)
        rs.set_state(state)
        for i, s in enumerate(_sets(nnv, rs, hw, cin)):       # fresh handles: nothing left over from the array
            net.reach(s, opts)
            for li, out in enumerate(net.reachSet):
                (lb, ub), V = got[li][i]
                elb, eub = out.estimateRanges()
                if li < 2 * len(convs):                        # (the FC layer's product splits by the size of the call)
                    assert np.array_equal(lb, elb) and np.array_equal(ub, eub) and np.array_equal(V, np.array(out.V)), (li, i)
                else:
                    scale = np.abs(out.V).max()
                    assert np.abs(V - np.array(out.V)).max() <= 1e-13 * scale and max(np.abs(lb - elb).max(), np.abs(ub - eub).max()) <= 1e-12 * scale * V.shape[-1]
    finally:
        ctx.set_switch("poison_pending", was)
