"""Arrays of boxes of unlike widths through two large layers: the second contracts the rows of the first's weights as they are and
multiplies by each set's scales on the way.  Against the dense product with what the ReLU step returned; one index list for all sets,
sixteen (sets with dimensions without width have lists of their own) and seventeen, which are too many; one whole tile of 128 columns, two and
ragged ones.  The sets that took the route are counted.  Bound: K + 4 rounded terms an entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


# (flat: so many sets have no width in their first three dimensions)
@pytest.mark.parametrize("n_in,hidden,out,count,flat", [(127, 300, 260, 86, 0), (128, 384, 257, 64, 0), (255, 300, 400, 66, 15), (255, 300, 400, 66, 16),
                                                        (130, 300, 400, 66, 15), (300, 513, 300, 64, 0), (127, 300, 260, 70, 0)])
def test_each_set_its_own_scales(nnv, n_in, hidden, out, count, flat):
    rs = np.random.RandomState(n_in)
    W1, b1 = rs.randn(hidden, n_in) / np.sqrt(n_in), rs.randn(hidden)
    W2, b2 = rs.randn(out, hidden) / np.sqrt(hidden), rs.randn(out)
    half = rs.rand(n_in, count) * 2e-2
    half[:3, 1:2 * flat:2] = 0.0
    x = rs.rand(n_in, count)
    opts = ("relax-star-area", [], 1, None, "linprog")
    S = nnv.Star.from_boxes(np.asfortranarray(x - half), np.asfortranarray(x + half))
    mid = nnv.layers.ReluLayer().reach(nnv.layers.FullyConnectedLayer(W1, b1).reach(S, *opts), *opts)
    ctx = S[0].ctx
    before = ctx.routes()["fc_scaled"]
    res = nnv.layers.FullyConnectedLayer(W2, b2).reach(mid, *opts)
    # (seventeen lists are packed set by set; fewer than 256 tiles of 128 x 128 are cut into narrower ones, which are packed too)
    wide = sum(-(-(n_in + 1 - (3 if i % 2 and i < 2 * flat else 0)) // 128) for i in range(count)) * -(-(-(-out // 16) * 16) // 128) >= 256
    assert ctx.routes()["fc_scaled"] - before == (count if wide and flat < 16 else 0)
    lbs, ubs = nnv.Star.estimateRanges_array(res)
    for i in (0, 1, 2, count // 2, count - 2, count - 1):
        Vin, V, plb, pub = np.array(mid[i].V), np.array(res[i].V), res[i].predicate_lb, res[i].predicate_ub
        exp = W2 @ Vin
        exp[:, 0] += b2
        tol = (hidden + 4) * EPS * (np.abs(W2) @ np.abs(Vin))
        tol[:, 0] += 4 * EPS * np.abs(b2)
        assert np.all(np.abs(V - exp) <= tol), i
        G, big = V[:, 1:], np.maximum(np.abs(plb), np.abs(pub))
        elb = V[:, 0] + np.maximum(G, 0) @ plb + np.minimum(G, 0) @ pub
        eub = V[:, 0] + np.maximum(G, 0) @ pub + np.minimum(G, 0) @ plb
        rtol = (V.shape[1] + hidden + 8) * EPS * (np.abs(V[:, 0]) + (np.abs(W2) @ np.abs(Vin[:, 1:])) @ big)
        assert np.all(np.abs(lbs[:, i] - elb) <= rtol) and np.all(np.abs(ubs[:, i] - eub) <= rtol), i
