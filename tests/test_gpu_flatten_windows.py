"""A C-style flatten of images that are in memory inside their windows only (the output of a pooling or convolution) against the
same network with every image written in full: a permutation of rows, the same to the bit.  Image sizes around multiples of 32 rows,
one channel and many; four columns a step (up to 1024 rows), two (up to 3968) and one, with an odd number of columns over two.  What nobody
wrote is poisoned, and that the images were read inside their windows is counted."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


@pytest.mark.parametrize("hw,cin,cout,pool", [((6, 5), 1, 1, 0), ((8, 8), 1, 4, 0), ((16, 16), 3, 16, 2), ((11, 13), 2, 7, 0), ((32, 32), 1, 4, 0),
                                              ((33, 31), 1, 4, 3), ((41, 25), 2, 1, 0), ((26, 40), 2, 1, 0), ((16, 31), 1, 8, 0), ((21, 21), 1, 9, 0)])
def test_flatten_inside_windows(nnv, hw, cin, cout, pool):
    rs = np.random.RandomState(hw[0] * cout)
    layers = [{"type": "conv", "W": rs.randn(3, 3, cin, cout), "b": rs.randn(cout), "padding": [1] * 4, "stride": [1, 1], "dilation": [1, 1]},
              {"type": "batchnorm", "mean": rs.randn(cout), "var": rs.rand(cout) + 0.5, "eps": 1e-5, "scale": rs.rand(cout) + 0.5, "offset": rs.randn(cout)}]
    if pool:
        layers.append({"type": "avgpool", "pool": [pool, pool], "stride": [pool, pool], "padding": [0] * 4})
    layers.append({"type": "flatten", "flatten_type": "nnet.keras.layer.FlattenCStyleLayer"})
    x = rs.rand(*hw, cin)
    ctx = nnv.default_context()

    def run():
        net = nnv.NN.from_config(layers)
        out = net.reach(nnv.ImageStar(x - 0.01, x + 0.01), {"reachMethod": "relax-star-area", "relaxFactor": 1})
        return np.array(out.V).reshape(-1, order="F"), [np.asarray(v).reshape(-1) for v in out.estimateRanges()], np.array(net.reachSet[-2].V)

    poisoned = ctx.switches["poison_pending"]
    ctx.set_switch("poison_pending", True)
    taken = ctx.routes()["permute_window"]
    try:
        V, r, before = run()
    finally:
        ctx.set_switch("poison_pending", poisoned)
    assert ctx.routes()["permute_window"] == taken + 1
    was = ctx.switches["no_conv_boxes"]
    ctx.set_switch("no_conv_boxes", True)
    try:
        Vd, rd, beford = run()
    finally:
        ctx.set_switch("no_conv_boxes", was)
    assert ctx.routes()["permute_window"] == taken + 1
    # (the convolution's and the range estimate's own sums may run in another order: fewer than 400 terms of the results' size)
    assert np.array_equal(V == 0, Vd == 0) and np.all(np.abs(V - Vd) <= 1e-13 * np.abs(Vd).max())
    assert all(np.all(np.abs(a - b) <= 1e-13 * np.abs(b).max()) for a, b in zip(r, rd))
    H, W, C, n = before.shape
    assert np.array_equal(V, before.transpose(2, 1, 0, 3).reshape(H * W * C, n, order="F").reshape(-1, order="F"))
