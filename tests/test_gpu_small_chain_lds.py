"""The one-launch reach whose sets stay in the LDS (no layer wider than 64 neurons), against the oracle: one to four row tiles, column
tiles at their edges, every neuron crossing, none, no row kept, FC layers behind one another, a dense input set, the widest and
deepest networks that fit and the first that do not (those take the other kernel and must give the same).  Every case asserts
which kernel its sets took."""
import numpy as np
import pytest

from oracle import nnv_oracle
from tests import test_gpu_small_chain
from tests.test_gpu_small_chain import _fc, _net

pytestmark = pytest.mark.gpu
AREA = "relax-star-area"


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    nnv_amd.default_context()
    return nnv_amd


def _check_against_oracle(nnv, oracle, layers, dev_in, ora_in, method, in_lds=True):
    ctx = nnv.default_context()
    before = ctx.routes()
    test_gpu_small_chain._check_against_oracle(nnv, oracle, layers, dev_in, ora_in, method)
    if not ctx.switch_is_on("no_small_chain", "dense_affine"):
        count = len(ora_in) if isinstance(ora_in, list) else 1
        took = {r: n - before[r] for r, n in ctx.routes().items() if r in ("chain", "chain_lds")}
        assert took == {"chain_lds": count if in_lds else 0, "chain": 0 if in_lds else count}


@pytest.mark.parametrize("widths,eps", [
    ((1, 1, 1), 0.5), ((2, 16, 16, 16), 0.3), ((5, 17, 32, 33, 2), 0.1), ((15, 48, 49, 1), 0.05), ((64, 64, 64, 64), 0.01), ((63, 63, 47, 64), 0.2),
    ((5, 50, 50, 50, 50, 50, 50, 5), 1.0), ((5, 50, 50, 50, 50, 50, 50, 5), 0.02), ((6, 50, 50, 50, 50, 50, 50, 5), 0.05),
    ((5, 64, 64, 64, 9), 0.7), ((5, 64, 64, 64, 64, 9), 0.2), ((31, 16, 16, 16, 16, 16, 16, 16, 16), 0.2)])
@pytest.mark.parametrize("method", ["relax-star-area", "relax-star-range", "relax-star-random"])
def test_widths(nnv, widths, eps, method):
    rs = np.random.RandomState(sum(widths))
    c = rs.rand(widths[0]) - 0.5
    _check_against_oracle(nnv, nnv_oracle, _net(rs, widths), nnv.Star(c - eps, c + eps), nnv_oracle.star_from_box(c - eps, c + eps), method)


# by the memory of the sets in front of the last layers (160 KB of LDS), the width of a layer (64), the columns of a layer (256)
@pytest.mark.parametrize("widths,n,in_lds", [
    ((34, 50, 50, 50, 50, 50, 50, 5), 34, True), ((35, 50, 50, 50, 50, 50, 50, 5), 35, False), ((5, 64, 64, 64, 64, 9), 5, True),
    ((5, 64, 64, 64, 64, 64, 9), 5, False), ((5, 50, 50, 50, 50, 50, 50, 50, 5), 5, False), ((64, 64, 64, 3), 64, True), ((65, 64, 64, 3), 65, False),
    ((8, 65, 40, 3), 8, False), ((8, 50, 4), 255, True), ((8, 50, 4), 256, False), ((8, 30, 4), 511, True), ((8, 30, 4), 512, False)])
def test_the_last_that_fit_and_the_first_that_do_not(nnv, widths, n, in_lds):
    rs = np.random.RandomState(n + len(widths))
    V = np.concatenate([rs.rand(widths[0], 1) - 0.5, rs.randn(widths[0], n) * (0.2 / n)], axis=1)
    args = (V, np.zeros((1, n)), np.zeros(1), -np.ones(n), np.ones(n))
    _check_against_oracle(nnv, nnv_oracle, _net(rs, widths), nnv.Star(*args), nnv_oracle.OStar(*args), AREA, in_lds)


@pytest.mark.parametrize("bias", [-30.0, 30.0, 0.0])
def test_no_row_kept_every_row_kept_every_row_crossing(nnv, bias):
    rs = np.random.RandomState(3)
    layers = _net(rs, (7, 45, 33, 20, 4))
    layers[2]["b"] = rs.randn(33) * 0.1 + bias
    c = np.zeros(7)
    eps = 0.3 if bias else 40.0
    _check_against_oracle(nnv, nnv_oracle, layers, nnv.Star(c - eps, c + eps), nnv_oracle.star_from_box(c - eps, c + eps), AREA)


def test_layers_in_other_orders_and_a_dense_input(nnv):
    rs = np.random.RandomState(4)
    V = rs.randn(12, 40)
    plb, pub = -rs.rand(39), rs.rand(39)
    args = (V, np.zeros((1, 39)), np.zeros(1), plb, pub)
    layers = [_fc(rs, 20, 12), _fc(rs, 41, 20), {"type": "relu"}, _fc(rs, 64, 41), {"type": "relu"}, _fc(rs, 3, 64), _fc(rs, 18, 3), {"type": "relu"}]
    _check_against_oracle(nnv, nnv_oracle, layers, nnv.Star(*args), nnv_oracle.OStar(*args), AREA)


def test_equal_keys_keep_their_order(nnv):
    """Every neuron twice: equal sort keys, smaller neuron first."""
    rs = np.random.RandomState(6)
    W, b = rs.randn(24, 5), np.zeros(24)
    layers = [{"type": "fc", "W": np.repeat(W, 2, axis=0), "b": np.repeat(b, 2)}, {"type": "relu"}, _fc(rs, 5, 48)]
    c = np.zeros(5)
    _check_against_oracle(nnv, nnv_oracle, layers, nnv.Star(c - 0.5, c + 0.5), nnv_oracle.star_from_box(c - 0.5, c + 0.5), AREA)


@pytest.mark.parametrize("count", [2, 200, 600])
def test_arrays(nnv, count):
    rs = np.random.RandomState(count)
    layers = _net(rs, (6, 50, 38, 5))
    lbs = rs.randn(6, count) * 0.3
    ubs = lbs + 0.4 * rs.rand(6, count) * (rs.rand(6, count) < 0.8)
    _check_against_oracle(nnv, nnv_oracle, layers, nnv.Star.from_boxes(lbs, ubs), [nnv_oracle.star_from_box(lbs[:, i], ubs[:, i]) for i in range(count)],
                          AREA)
