"""Boxes whose host arrays are large enough to be shared out to the context's threads (1.5 MB), or just not: the same sets, to the
bit, as boxes made one by one; half-widths all alike, alike in all but a few sets, all different, zero in some dimensions, parts
that end inside a set and inside the copied pieces; and the private copies of the bounds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


@pytest.mark.parametrize("N,count", [(131, 1000), (132, 1001), (1031, 129), (785, 1400), (4, 35000), (17, 9000),
                                     (196, 1003), (197, 1001), (1031, 193), (4, 50000), (22, 9000)])
@pytest.mark.parametrize("widths", ["alike", "few", "different", "degenerate"])
def test_boxes_of_large_arrays(nnv, N, count, widths):
    rs = np.random.RandomState(N + count)
    half = np.repeat((rs.randint(1, 9, N) / 16.0)[:, None], count, axis=1)
    if widths == "few":
        for i in rs.choice(count, 5, replace=False):
            half[rs.randint(N), i] = 2.0
    elif widths == "different":
        half = rs.randint(1, 1 << 20, (N, count)) / 1024.0
    elif widths == "degenerate":
        half[rs.rand(N) < 0.3] = 0.0
    centre = rs.randint(-64, 64, (N, count)) / 32.0
    lb, ub = np.asfortranarray(centre - half), np.asfortranarray(centre + half)
    sets = nnv.Star.from_boxes(lb, ub)
    klb, kub = lb.copy(), ub.copy()
    lb[:] = 0.0                                               # (the sets keep copies of their own)
    ub[:] = 0.0
    llb, lub = nnv.Star.estimateRanges_array(sets)
    assert np.array_equal(llb, klb) and np.array_equal(lub, kub)
    for i in sorted({0, 1, count // 3, count - 1}):
        one = nnv.Star(klb[:, i], kub[:, i])
        assert sets[i].nVar == one.nVar and np.array_equal(sets[i].V, one.V)
        assert np.array_equal(sets[i].state_lb, klb[:, i]) and np.array_equal(sets[i].state_ub, kub[:, i])


def test_without_threads(nnv):
    ctx = nnv.default_context()
    was = ctx.switch_is_on("no_host_pool")
    ctx.set_switch("no_host_pool", True)
    try:
        test_boxes_of_large_arrays(nnv, 785, 1400, "few")
    finally:
        ctx.set_switch("no_host_pool", was)
