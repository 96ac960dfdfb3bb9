"""A fully connected layer of few outputs straight behind a ReLU step (one launch over the rows the step kept and the unit vectors it
appended) against the dense product with the step's whole matrix, at the edges of its tiles: 16 columns a tile, 128 unit vectors a
block, 1024 kept rows at a time, 16 and 32 outputs; no row kept, no neuron crossing, nothing but the centre; columns of the layer
before that nobody has written; arrays.  Bound: an entry is a sum of at most K + 2 rounded products, |error| <= (K + 4) eps |W| |V|; a
range is a sum of n + 1 such terms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _relu(nnv, S):
    return nnv.layers.ReluLayer().reach(S, "relax-star-area", [], 1, None, "linprog")


def _fc(nnv, S, W, b):
    return nnv.layers.FullyConnectedLayer(W, b).reach(S, "relax-star-area", [], 1, None, "linprog")


def _check(mid, out, W, b, what):
    """mid: what the ReLU step returned, read after the layer has run on it."""
    Vin, V, plb, pub = np.array(mid.V), np.array(out.V), out.predicate_lb, out.predicate_ub
    exp = W @ Vin
    exp[:, 0] += b
    tol = (W.shape[1] + 4) * EPS * (np.abs(W) @ np.abs(Vin))
    tol[:, 0] += 4 * EPS * np.abs(b)
    assert V.shape == exp.shape and np.all(np.abs(V - exp) <= tol), what
    G, big = V[:, 1:], np.maximum(np.abs(plb), np.abs(pub))
    lb, ub = out.estimateRanges()
    elb = V[:, 0] + np.maximum(G, 0) @ plb + np.minimum(G, 0) @ pub
    eub = V[:, 0] + np.maximum(G, 0) @ pub + np.minimum(G, 0) @ plb
    rtol = (V.shape[1] + 8) * EPS * (np.abs(V[:, 0]) + np.abs(G) @ big)
    assert np.all(np.abs(lb - elb) <= rtol) and np.all(np.abs(ub - eub) <= rtol), what


def _star(nnv, rs, K, n, kept, crossing):
    """K rows of which `kept` stay, `crossing` cross zero and the others are reset, in random places; n generators."""
    V = rs.randn(K, n + 1) / (4.0 * n)
    V[:, 0] = np.repeat([2.0, 0.0, -2.0], [kept, crossing, K - kept - crossing])
    return nnv.Star(np.asfortranarray(V[rs.permutation(K)]), np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n))


@pytest.mark.parametrize("M,K,n,kept,crossing", [
    (1, 20, 15, 7, 6), (10, 100, 16, 1, 99), (16, 100, 14, 0, 60), (17, 130, 31, 130, 0), (32, 300, 47, 33, 128), (5, 300, 200, 32, 129),
    (10, 1100, 33, 1024, 1), (32, 1500, 20, 1030, 2), (3, 2100, 5, 2049, 16), (2, 3, 1, 3, 0), (10, 50, 30, 0, 0)])
def test_outputs_and_ranges(nnv, M, K, n, kept, crossing):
    rs = np.random.RandomState(M + 3 * K + n)
    W, b = rs.randn(M, K), rs.randn(M)
    S = _star(nnv, rs, K, n, kept, crossing)
    before = S.ctx.routes()["fc_skinny"]
    mid = _relu(nnv, S)
    out = _fc(nnv, mid, W, b)
    assert S.ctx.routes()["fc_skinny"] == before + 1
    _check(mid, out, W, b, "one set")


@pytest.mark.parametrize("count", [1, 3])
def test_behind_unwritten_columns(nnv, count):
    """Two large layers in front: the columns the second gathered are described, not in memory."""
    rs = np.random.RandomState(count)
    W1, W2, W3 = rs.randn(300, 200) / 14, rs.randn(257, 300) / 17, rs.randn(9, 257)
    b1, b2, b3 = rs.randn(300), 0.1 * rs.randn(257), rs.randn(9)
    x = rs.rand(200, count)
    S = nnv.Star.from_boxes(np.asfortranarray(x - 0.02), np.asfortranarray(x + 0.02)) if count > 1 else nnv.Star(x[:, 0] - 0.02, x[:, 0] + 0.02)
    mid = _relu(nnv, _fc(nnv, _relu(nnv, _fc(nnv, S, W1, b1)), W2, b2))
    ctx = (S if count == 1 else S[0]).ctx
    before = ctx.routes()["fc_skinny"]
    out = _fc(nnv, mid, W3, b3)
    assert ctx.routes()["fc_skinny"] == before + count
    for i in range(count):
        _check(mid if count == 1 else mid[i], out if count == 1 else out[i], W3, b3, "set %d" % i)


def test_infinite_weight_takes_the_dense_product(nnv):
    """An infinite weight times the zero of a reset row is NaN."""
    rs = np.random.RandomState(5)
    W, b = rs.randn(4, 60), rs.randn(4)
    W[2, 7] = np.inf
    S = _star(nnv, rs, 60, 12, 20, 20)
    before = S.ctx.routes()["fc_skinny"]
    mid = _relu(nnv, S)
    out = _fc(nnv, mid, W, b)
    assert S.ctx.routes()["fc_skinny"] == before
    with np.errstate(invalid="ignore"):
        assert np.array_equal(np.isnan(np.array(out.V)), np.isnan(W @ np.array(mid.V)))


@pytest.mark.parametrize("hint", [True, False])
def test_no_product_of_range_sums_is_formed_for_it(nnv, hint):
    """An inner layer of few outputs over an array large enough for one: the kernel sums its columns itself.  The layer behind it
    is not of few outputs; its product is formed once, whether the ReLU step is told of the layer or not, and read."""
    rs = np.random.RandomState(17)
    count, widths = 64, [40, 256, 24, 240]
    fcs = [nnv.layers.FullyConnectedLayer(rs.randn(m, k) / np.sqrt(k), 0.1 * rs.randn(m)) for k, m in zip(widths, widths[1:])]
    opts = ("relax-star-area", [], 1, None, "linprog")
    x = rs.rand(40, count)
    s = fcs[0].reach(nnv.Star.from_boxes(np.asfortranarray(x - 0.3), np.asfortranarray(x + 0.3)), *opts)
    ctx = s[0].ctx
    for layer, formed, skinny in ((fcs[1], 0, count), (fcs[2], count, 0)):
        was = ctx.routes()
        if hint:
            ctx.hint_next_fc(layer._weights(ctx))
        mid = nnv.layers.ReluLayer().reach(s, *opts)
        s = layer.reach(mid, *opts)
        now = ctx.routes()
        assert [now[k] - was[k] for k in ("sums_product", "sums_product_read", "fc_skinny")] == [formed, formed, skinny]
        for i in (0, count - 1):
            _check(mid[i], s[i], np.asarray(layer.Weights), np.asarray(layer.Bias).reshape(-1), (layer.OutputSize, i))


@pytest.mark.parametrize("last", [10, 40])
def test_a_reach_forms_no_product_that_nobody_reads(nnv, last):
    """The last layer writes its columns whoever forms their sums: the ReLU step in front of it is not told of it."""
    rs = np.random.RandomState(last)
    count, widths = 64, [40, 256, 240, last]
    layers = []
    for k, m in zip(widths, widths[1:]):
        layers += [{"type": "fc", "W": rs.randn(m, k) / np.sqrt(k), "b": 0.1 * rs.randn(m)}, {"type": "relu"}]
    net = nnv.NN.from_config(layers[:-1])
    x = rs.rand(40, count)
    S = nnv.Star.from_boxes(np.asfortranarray(x - 0.3), np.asfortranarray(x + 0.3))
    ctx = S[0].ctx
    was = ctx.routes()
    out = net.reach(S, {"reachMethod": "relax-star-area", "relaxFactor": 1})
    now = ctx.routes()
    # the first layer's, over the boxes, and the second's
    assert [now[k] - was[k] for k in ("sums_product", "sums_product_read")] == [2 * count, 2 * count]
    for i in (0, count - 1):
        _check(net.reachSet[3][i], out[i], layers[-2]["W"], layers[-2]["b"], i)
