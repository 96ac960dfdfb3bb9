"""Ranges of a fully connected layer's output whose sums come partly from the product's tiles, at the number of tiles a block asks for
ahead: 32 and 33, 128 and 129 tiles of 128 columns; 66 and 18 row blocks (dealt to the XCDs in rounds of 72 and 24); narrower
tiles.  The route is counted, and where the sums of more than 32 tiles are asked for ahead.  The bound is that of the ranges of few
rows: n + K + 16 rounded terms."""
import numpy as np
import pytest

from tests.test_gpu_final_rows import _check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


# (enough crossing neurons for the layer's columns of them to be worth a route of their own: M K crossing >= 4e6 padded)
@pytest.mark.parametrize("M,K,n,many", [(520, 260, 4095, 0), (520, 260, 4096, 1), (136, 520, 16383, 1), (136, 520, 16384, 1), (136, 520, 2047, None),
                                        (136, 520, 8191, 1)])
def test_many_tiles_of_sums(nnv, M, K, n, many):
    rs = np.random.RandomState(n)
    W, b = rs.randn(M, K) / np.sqrt(K), rs.randn(M)
    V = rs.randn(K, n + 1) * (0.5 / n)
    V[:, 0] = rs.choice([-2.0, 0.0, 2.0], K)
    S = nnv.Star(V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n))
    opts = ("relax-star-area", [], 1, None, "linprog")
    was = S.ctx.routes()
    mid = nnv.layers.ReluLayer().reach(S, *opts)
    out = nnv.layers.FullyConnectedLayer(W, b).reach(mid, *opts)
    now = S.ctx.routes()
    assert now["fc_rowsum"] == was["fc_rowsum"] + 1
    if many is not None:
        assert now["fc_rowsum_many"] == was["fc_rowsum_many"] + many
    _check(out, W, np.array(mid.V), "behind a ReLU step")
