"""Ranges of outputs of few rows over many columns (the sums of many column chunks are combined by sixteen waves to 16 rows), and of
layers whose sums come straight from the weights, at the edges: chunks one below and at the rule, 16 and 17 rows, more tiles than a
block asks for ahead.  Bound: a range is a sum of n + 1 rounded terms, |error| <= (n + 4) eps (|c| + sum |v| max(|plb|, |pub|)) entry
by entry, and the entries themselves are products of K terms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _check(o, W, Vin, what):
    lb, ub = o.estimateRanges()
    V, plb, pub = np.array(o.V), o.predicate_lb, o.predicate_ub
    G = V[:, 1:]
    elb = V[:, 0] + np.maximum(G, 0) @ plb + np.minimum(G, 0) @ pub
    eub = V[:, 0] + np.maximum(G, 0) @ pub + np.minimum(G, 0) @ plb
    big = np.maximum(np.abs(plb), np.abs(pub))
    tol = (G.shape[1] + 8) * EPS * (np.abs(V[:, 0]) + np.abs(G) @ big) + (W.shape[1] + 8) * EPS * (np.abs(W) @ (np.abs(Vin[:, 1:]) @ big + np.abs(Vin[:, 0])))
    assert np.all(np.abs(lb - elb) <= tol) and np.all(np.abs(ub - eub) <= tol), what


@pytest.mark.parametrize("rows,n", [(1, 400), (10, 1023), (16, 1024), (16, 1100), (17, 1090), (33, 2200), (64, 5000), (10, 20000)])
def test_few_rows_many_columns(nnv, rows, n):
    rs = np.random.RandomState(rows + n)
    V = rs.randn(40, n + 1)
    S = nnv.Star(V, np.zeros((1, n)), np.zeros(1), -rs.rand(n), rs.rand(n))
    W, b = rs.randn(rows, 40), rs.randn(rows)
    _check(S.affineMap(W, b), W, V, "map")


@pytest.mark.parametrize("M,K,n", [(128, 200, 300), (136, 1000, 33), (520, 1030, 700), (130, 300, 2300), (2048, 2000, 40)])
def test_sums_from_the_weights(nnv, M, K, n):
    rs = np.random.RandomState(M + K)
    W, b = rs.randn(M, K) / np.sqrt(K), rs.randn(M)
    x = rs.rand(K)
    box = nnv.Star(x - 0.1, x + 0.1)
    _check(box.affineMap(W, b), W, np.array(box.V), "box")
    V = rs.randn(K, n + 1) * 0.05
    V[:, 0] += rs.choice([-0.6, 0.0, 0.6], K)
    S = nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n))
    mid = nnv.layers.ReluLayer().reach(S, "relax-star-area", [], 1, None, "linprog")
    out = nnv.layers.FullyConnectedLayer(W, b).reach(mid, "relax-star-area", [], 1, None, "linprog")
    _check(out, W, np.array(mid.V), "behind a ReLU step")
