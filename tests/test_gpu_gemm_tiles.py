"""Products of a fully connected layer at the edges of their tiles (32 and 64 rows and columns, 16 rows for small outputs) and of their
stages (16 and 32 rows of the contraction, one stage more or fewer than the ring holds, split contractions): the plain
product, the one over the rows a ReLU step kept, and the one of an array, against numpy in the widest type it has.  Bound: the
contraction and the bias add K + 1 rounded terms, |error| <= (K + 2) eps |W| |V| entry by entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _star(nnv, rs, K, n):
    V = rs.randn(K, n + 1)
    return nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n)), V


def _check(got, W, b, V, what):
    exp = (W.astype(np.longdouble) @ V.astype(np.longdouble)).astype(np.longdouble)
    exp[:, 0] += b
    bound = (W.shape[1] + 2) * EPS * (np.abs(W) @ np.abs(V) + (np.arange(V.shape[1]) == 0) * np.abs(b)[:, None])
    assert got.shape == exp.shape, what
    assert np.all(np.abs(got - exp) <= bound), what


# M (rows of the output), K (contraction), n (generators)
SIZES = [(1, 1, 1), (15, 33, 62), (16, 16, 63), (17, 17, 64), (31, 31, 65), (32, 47, 127), (33, 48, 31), (63, 63, 30), (64, 64, 32), (65, 65, 33),
         (80, 129, 95), (96, 128, 96), (130, 255, 40), (257, 96, 300), (300, 700, 1030), (1030, 1040, 1100), (700, 2100, 70), (40, 2500, 2000)]


@pytest.mark.parametrize("M,K,n", SIZES)
def test_plain_product(nnv, M, K, n):
    rs = np.random.RandomState(M + K + n)
    S, V = _star(nnv, rs, K, n)
    W, b = rs.randn(M, K), rs.randn(M)
    out = S.affineMap(W, b)
    lb, ub = out.estimateRanges()
    got = np.array(out.V)
    _check(got, W, b, V, "V")
    half = np.abs(got[:, 1:]).sum(1)
    tol = (n + 4) * EPS * (half + np.abs(got[:, 0]))
    assert np.all(np.abs(lb - (got[:, 0] - half)) <= tol) and np.all(np.abs(ub - (got[:, 0] + half)) <= tol)


@pytest.mark.parametrize("count", [1, 3, 70])
@pytest.mark.parametrize("M,K,n", [(20, 300, 40), (129, 300, 70), (200, 333, 129), (257, 700, 64), (512, 600, 300)])
def test_product_over_kept_rows(nnv, count, M, K, n):
    if count == 70 and M * n > 40000:
        pytest.skip("covered by the smaller arrays")
    rs = np.random.RandomState(M + K + n + count)
    sets = []
    for i in range(count):
        V = rs.randn(K, n + 1) * 0.02
        V[:, 0] += rs.randn(K) * (0.2 + 0.1 * (i % 3))   # some rows pass, some cross, some are reset
        sets.append(nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n)))
    W, b = rs.randn(M, K), rs.randn(M)
    L = [nnv.layers.ReluLayer(), nnv.layers.FullyConnectedLayer(W, b)]
    mid = L[0].reach(sets if count > 1 else sets[0], "relax-star-area", [], 1, None, "linprog")
    out = L[1].reach(mid, "relax-star-area", [], 1, None, "linprog")
    for i in sorted({0, count // 2, count - 1}):
        m, o = (mid[i], out[i]) if count > 1 else (mid, out)
        lb, ub = o.estimateRanges()
        got, V = np.array(o.V), np.array(m.V)
        _check(got, W, b, V, "set %d" % i)
        plb, pub = o.predicate_lb, o.predicate_ub
        G = got[:, 1:]
        elb = got[:, 0] + np.maximum(G, 0) @ plb + np.minimum(G, 0) @ pub
        eub = got[:, 0] + np.maximum(G, 0) @ pub + np.minimum(G, 0) @ plb
        # (the sums may be formed from the weights and the columns' scales instead of from the rounded columns)
        tol = (G.shape[1] + 8) * EPS * (np.abs(got[:, 0]) + np.abs(G) @ np.maximum(np.abs(plb), np.abs(pub))) + (K + 8) * EPS * (
            np.abs(W) @ (np.abs(V[:, 1:]) @ np.maximum(np.abs(plb), np.abs(pub))))
        assert np.all(np.abs(lb - elb) <= tol) and np.all(np.abs(ub - eub) <= tol), "ranges of set %d" % i


@pytest.mark.parametrize("kept", [1023, 1024, 2016, 2048, 2049, 3072, 3088, 5000])
@pytest.mark.parametrize("M,n", [(20, 30), (150, 70), (520, 300)])
def test_long_lists_of_kept_rows(nnv, kept, M, n):
    """The numbers of the kept rows go through LDS 2048 at a time, half by half; few output rows and columns split the contraction."""
    rs = np.random.RandomState(kept + M)
    K = kept + kept // 3
    V = rs.randn(K, n + 1) * 0.01
    V[:, 0] = -2.0 * n
    V[np.sort(rs.permutation(K)[:kept]), 0] *= -1.0
    S = nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n))
    W, b = rs.randn(M, K), rs.randn(M)
    mid = nnv.layers.ReluLayer().reach(S, "relax-star-area", [], 1, None, "linprog")
    out = nnv.layers.FullyConnectedLayer(W, b).reach(mid, "relax-star-area", [], 1, None, "linprog")
    got = np.array(out.V)
    keep = V[:, 0] > 0
    assert mid.nVar == n and keep.sum() == kept
    _check(got, W[:, keep], b, V[keep], "kept %d" % kept)


@pytest.mark.parametrize("M,share", [(150, 0.7), (24, 0.7), (150, 0.3)])
def test_long_lists_in_an_array(nnv, M, share):
    """The same for the sets of an array, each with a list of its own, longer or shorter than what LDS holds at a time."""
    rs = np.random.RandomState(M)
    n, H, count = 30, 4500, 12
    c = rs.rand(n, count)
    h = 0.001 * rs.rand(n, count)
    L1 = nnv.layers.FullyConnectedLayer(rs.randn(H, n) * 0.1, np.where(rs.rand(H) < share, 3.0, -3.0) + 0.2 * rs.randn(H))
    mid = nnv.layers.ReluLayer().reach(L1.reach(nnv.Star.from_boxes(c - h, c + h), "relax-star-area", [], 1, None, "linprog"), "relax-star-area", [],
                                       1, None, "linprog")
    W, b = rs.randn(M, H), rs.randn(M)
    out = nnv.layers.FullyConnectedLayer(W, b).reach(mid, "relax-star-area", [], 1, None, "linprog")
    for i in (0, 5, count - 1):
        Vm = np.array(mid[i].V)
        keep = np.any(Vm != 0, axis=1)
        assert (keep.sum() > 2048) == (share > 0.5)
        _check(np.array(out[i].V), W[:, keep], b, Vm[keep], "set %d" % i)


@pytest.mark.parametrize("M", [(1 << 24) - 16, 1 << 24])
def test_offsets_at_the_end_of_32_bits(nnv, M):
    """Leading dimensions of W on both sides of the line behind which offsets have 64 bits.  Small whole numbers: exact."""
    from nnv_amd import _lib
    K = 3
    rs = np.random.RandomState(M % 97)
    n = 4
    ctx = _lib.Context(0)
    W = np.asfortranarray(rs.randint(-3, 4, (M, K)).astype(np.float64))
    b = rs.randint(-3, 4, M).astype(np.float64)
    V = np.asfortranarray(rs.randint(-3, 4, (K, n + 1)).astype(np.float64))
    S = nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n), ctx=ctx)
    out = S.affineMap(W, b)
    lb, ub = out.estimateRanges()
    P = W @ V
    half = np.abs(P[:, 1:]).sum(1)
    assert np.array_equal(lb, P[:, 0] + b - half) and np.array_equal(ub, P[:, 0] + b + half)


def test_infinite_weight_meets_no_padding(nnv):
    """Rows a list is padded with are no rows of the set: an infinite weight in column 0 does not reach them."""
    rs = np.random.RandomState(3)
    K, n, M = 300, 40, 150
    V = rs.randn(K, n + 1) * 0.02
    V[:, 0] = np.where(rs.rand(K) < 0.3, 1.0, -1.0)
    V[0, 0] = -1.0                                        # row 0 is reset
    W, b = rs.randn(M, K), rs.randn(M)
    W[5, 0] = np.inf
    S = nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n))
    mid = nnv.layers.ReluLayer().reach(S, "relax-star-area", [], 1, None, "linprog")
    out = nnv.layers.FullyConnectedLayer(W, b).reach(mid, "relax-star-area", [], 1, None, "linprog")
    got, Vm = np.array(out.V), np.array(mid.V)
    keep = np.any(Vm != 0, axis=1)
    _check(np.delete(got, 5, 0), np.delete(W, 5, 0)[:, keep], np.delete(b, 5), Vm[keep], "finite rows")
    assert np.all(np.isfinite(np.delete(got, 5, 0)))
