"""Sets made one after the other: their bounds are fetched several sets at a time (the first at once, up to sixteen later ones with the
next call that is not a constructor).  Whatever comes in between - sets that are dropped at once, sizes that differ, a set too
large for it, a staging ring that wraps, a launch that fails - every set has its own centre and generators, to the bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _check(S, lb, ub):
    V = np.array(S.V)
    half = 0.5 * (ub - lb)
    keep = np.flatnonzero(half != 0) if lb.size > 1 else np.arange(1)
    exp = np.zeros((lb.size, keep.size + 1))
    exp[:, 0] = 0.5 * (lb + ub)
    exp[keep, 1 + np.arange(keep.size)] = half[keep]
    assert np.array_equal(V, exp)
    assert np.array_equal(S.predicate_lb, -np.ones(keep.size)) and np.array_equal(S.predicate_ub, np.ones(keep.size))


@pytest.mark.parametrize("count", [1, 2, 16, 17, 18, 40])
def test_runs_of_constructors(nnv, count):
    rs = np.random.RandomState(count)
    made = []
    ctx = nnv.default_context()
    ctx.synchronize()        # (nothing waits, and the first of the run goes at once)
    was = ctx.routes()
    for i in range(count):
        n = int(rs.choice([1, 2, 15, 16, 17, 300, 784]))
        lb = rs.randn(n)
        ub = lb + rs.rand(n) * (rs.rand(n) < 0.8)
        S = nnv.Star(lb, ub)
        if i % 3 == 1:
            del S            # its memory is free for the next one's only behind the copy that still goes there
            continue
        made.append((S, lb.copy(), ub.copy()))
        lb += 1.0            # the caller's arrays are its own again
        ub -= 7.0
    ctx.synchronize()
    now = ctx.routes()
    assert [now[k] - was[k] for k in ("copies_fetched", "copies_together")] == [count, count - 1]
    for S, lb, ub in made:
        _check(S, lb, ub)


@pytest.mark.parametrize("n,fetched", [(7280, 3), (7281, 0)])
def test_the_largest_piece_a_kernel_fetches(nnv, n, fetched):
    """256 KB: 262080 bytes of centre, half-widths, bounds and index list on one side of the line, 262656 on the other."""
    rs = np.random.RandomState(n)
    ctx = nnv.default_context()
    ctx.synchronize()
    was = ctx.routes()["copies_fetched"]
    made = []
    for _ in range(3):
        lb = rs.randn(n)
        ub = lb + 0.5 + rs.rand(n)
        made.append((nnv.Star(lb, ub), lb, ub))
    ctx.synchronize()
    assert ctx.routes()["copies_fetched"] == was + fetched
    for S, lb, ub in made:
        l, u = S.estimateRanges()
        tol = 4 * np.finfo(float).eps * (np.abs(lb) + np.abs(ub))
        assert np.all(np.abs(l - lb) <= tol) and np.all(np.abs(u - ub) <= tol)
        rows = S._h.fetch_rows([0, n - 1])
        assert rows[0, 1] == 0.5 * (ub[0] - lb[0]) and rows[1, n] == 0.5 * (ub[-1] - lb[-1]) and np.count_nonzero(rows[:, 1:]) == 2
        assert np.array_equal(S.predicate_lb, -np.ones(n)) and np.array_equal(S.predicate_ub, np.ones(n))


def test_large_and_small_in_turn_past_the_end_of_the_ring(nnv):
    rs = np.random.RandomState(9)
    for rep in range(4):
        made = []
        for n in [3000, 70000, 5, 120000, 64, 64, 20000]:
            lb = rs.randn(n)
            ub = lb.copy()
            ub[:: max(1, n // 40)] += 0.25     # few generators: the matrices stay small
            made.append((nnv.Star(lb, ub), lb, ub))
        for S, lb, ub in made:
            l, u = S.estimateRanges()
            tol = 4 * np.finfo(float).eps * (np.abs(lb) + np.abs(ub))
            assert np.all(np.abs(l - lb) <= tol) and np.all(np.abs(u - ub) <= tol)


def test_bounds_in_any_layout(nnv):
    """Strided, transposed, integer and read-only bounds: the set reads a copy."""
    a = np.arange(60.0).reshape(6, 10)
    ro = a[2].copy()
    ro.setflags(write=False)
    for lb in (a[:, 3], a.T[2], a[1, ::3], np.arange(5), ro, a[:, :1]):
        lbf = np.asarray(lb, dtype=np.float64)
        _check(nnv.Star(lb, lb + 2), lbf.reshape(-1), lbf.reshape(-1) + 2)


def _boxes(ctx, nnv, rs, count):
    made = []
    for n in rs.choice([1, 16, 17, 300], count):
        lb = rs.randn(int(n))
        ub = lb + rs.rand(lb.size)
        made.append((nnv.Star(lb, ub, ctx=ctx), lb, ub))
    return made


def test_bounds_whose_copy_could_not_be_launched_go_on_waiting(nnv):
    """The constructors have returned: every later call fails until the bounds are there, and then all is as if nothing had been."""
    from nnv_amd import _lib
    ctx, rs = _lib.Context(0), np.random.RandomState(3)
    for count in (2, 6, 16):   # one at once, the others wait
        made = _boxes(ctx, nnv, rs, count)
        ctx.debug_fail_copies(2)
        with pytest.raises(_lib.NNVHipError):
            made[-1][0].estimateRanges()
        with pytest.raises(_lib.NNVHipError):
            ctx.synchronize()
        for S, lb, ub in made:
            _check(S, lb, ub)


def test_a_constructor_that_cannot_launch_the_waiting_copies_fails_alone(nnv):
    from nnv_amd import _lib
    ctx, rs = _lib.Context(0), np.random.RandomState(4)
    made = _boxes(ctx, nnv, rs, 16)   # fifteen wait
    ctx.debug_fail_copies(2)
    for _ in range(2):                # the sixteenth that waits, and one that finds sixteen waiting
        with pytest.raises(_lib.NNVHipError):
            _boxes(ctx, nnv, rs, 1)
    made += _boxes(ctx, nnv, rs, 20)
    for S, lb, ub in made:
        _check(S, lb, ub)


def test_a_context_goes_with_copies_that_cannot_be_launched(nnv):
    from nnv_amd import _lib
    ctx = _lib.Context(0)
    made = _boxes(ctx, nnv, np.random.RandomState(5), 5)
    del made
    ctx.debug_fail_copies(100)
    _lib.check(ctx.lib.nnvhip_destroy(ctx.handle))
    ctx.handle = None
