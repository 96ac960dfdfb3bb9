"""Ranges of a fully connected layer's output whose sums come partly from the GEMM's tiles, at the number of tiles a block asks for
ahead: 32, 33, 128 and 129 tiles of 64 columns, 17 row blocks (dealt to the XCDs in a round of 24).  The bound is that of the
ranges of few rows: n + K + 16 rounded terms."""
import numpy as np
import pytest

from tests.test_gpu_final_rows import _check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


@pytest.mark.parametrize("n", [2047, 2048, 8191, 8192])
def test_many_tiles_of_sums(nnv, n):
    rs = np.random.RandomState(n)
    M, K = 136, 260
    W, b = rs.randn(M, K) / np.sqrt(K), rs.randn(M)
    V = rs.randn(K, n + 1) * (0.5 / n)
    V[:, 0] = rs.choice([-2.0, 0.0, 2.0], K)
    S = nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n))
    opts = ("relax-star-area", [], 1, None, "linprog")
    mid = nnv.layers.ReluLayer().reach(S, *opts)
    out = nnv.layers.FullyConnectedLayer(W, b).reach(mid, *opts)
    out.estimateRanges()
    _check(out, W, np.array(mid.V), "behind a ReLU step")
