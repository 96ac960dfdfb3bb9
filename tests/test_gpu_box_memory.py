"""What boxes and released arrays hold on to: a box array that could never be written whole is refused where it is made,
staging memory stays bounded whatever the array's size, and the queue of released arrays stays bounded in a loop."""
import ctypes as C
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nnv():
    import nnv_amd
    return nnv_amd


def _free_and_total():
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value, total.value


def test_a_box_that_fits_the_device_but_not_what_is_free_is_refused(nnv):
    """Star(lb, ub) writes no matrix, but one that no reader could be given is refused at once: an N x (N + 1) matrix a
    little smaller than the device's memory, part of which is always taken."""
    ctx = nnv.default_context()
    ctx.trim_pool()
    _, total = _free_and_total()
    N = int((total / 8.0) ** 0.5) // 16 * 16 - 16
    free, _ = _free_and_total()
    assert 8 * N * (N + 1) <= total
    if 8 * N * (N + 1) <= free:
        pytest.skip("nothing of the device's memory is taken")
    lb = np.zeros(N)
    with pytest.raises(MemoryError):
        nnv.Star(lb, lb + 1.0)
    s = nnv.Star(lb[:1000], lb[:1000] + 1.0)         # the context goes on
    assert np.array_equal(s.estimateRanges()[1], np.ones(1000))


@pytest.mark.parametrize("N,count", [(1500, 1100), (70001, 31), (1100000, 2)])
@pytest.mark.parametrize("shared", [True, False])
def test_large_box_arrays_travel_in_pieces(nnv, N, count, shared):
    """More bounds than one piece of the staging ring holds: centres, half-widths and index lists arrive whole, with sets
    that share their half-widths and sets that all have their own."""
    from nnv_amd import _lib
    rs = np.random.RandomState(N + count)
    ctx = _lib.Context(0)                             # (a context of its own: other tests may have grown the shared one's ring)
    x = rs.rand(N, count)
    w = np.where(rs.rand(N, 1 if shared else count) < 3.0 / N, rs.rand(N, 1 if shared else count), 0.0) * np.ones((1, count))
    lbs, ubs = x - w, x + w
    sets = nnv.Star.from_boxes(lbs, ubs, ctx=ctx)
    ring, outgrown = ctx.staging_bytes()
    assert ring <= 16 << 20 and outgrown <= ring
    lb, ub = nnv.Star.estimateRanges_array(sets)
    c, v = 0.5 * (lbs + ubs), 0.5 * (ubs - lbs)
    assert np.array_equal(lb, c - v) and np.array_equal(ub, c + v)
    for i in (0, count // 2, count - 1):
        nz = np.flatnonzero(v[:, i])
        assert sets[i].nVar == nz.size
        V = sets[i].V
        assert np.array_equal(V[:, 0], c[:, i]) and np.array_equal(V[nz, 1 + np.arange(nz.size)], v[nz, i])
        assert np.count_nonzero(V[:, 1:]) == nz.size
    del sets
    gc.collect()
    _lib.check(ctx.lib.nnvhip_destroy(ctx.handle))


def test_the_queue_of_released_arrays_stays_bounded(nnv):
    """A loop of reaches over an array of 300 sets: the handles of the passes before are let go, device memory is not asked
    for once per pass."""
    rs = np.random.RandomState(1)
    dims = [8, 100, 100, 100, 100, 100, 5]
    layers = []
    for a, b in zip(dims[:-1], dims[1:]):
        layers += [{"type": "fc", "W": rs.randn(b, a) * np.sqrt(2.0 / a), "b": rs.randn(b) * 0.1}, {"type": "relu"}]
    net = nnv.NN.from_config(layers[:-1])
    ctx = nnv.default_context()
    ctx.trim_pool()
    held = sum(ctx.pool_stats())
    x = rs.rand(8, 300)
    queued, mallocs = [], []
    for _ in range(120):
        out = net.reach(nnv.Star.from_boxes(x - 0.05, x + 0.05), {"reachMethod": "relax-star-area", "relaxFactor": 1})
        nnv.Star.estimateRanges_array(out)
        now = ctx.debug_counters()
        queued.append(now["deferred_handles"])
        mallocs.append(now["device_mallocs"])
    assert max(queued) <= 4096 + 3 * 12 * 300, queued
    # (which blocks are free when depends on how long the host waits, so a few are asked for now and then; a queue that only
    # grows asks for one or more per FC layer, three hundred and more in fifty passes)
    assert mallocs[-1] - mallocs[-51] < 50, mallocs
    assert sum(ctx.pool_stats()) - held < 8 << 30  # (0.2 GB a pass)


@pytest.mark.parametrize("N,count", [(1, 1), (7, 3), (130, 2), (784, 1)])
def test_a_box_matrix_is_read_without_being_written(nnv, N, count):
    """V of a box whose matrix nobody has needed on the device: read twice, in memory afterwards as little as before."""
    rs = np.random.RandomState(N)
    lbs = rs.randn(N, count)
    ubs = lbs + rs.rand(N, count) * (rs.rand(N, count) < 0.7)
    sets = nnv.Star.from_boxes(lbs, ubs)
    ctx = nnv.default_context()
    before = ctx.pool_stats()[0]
    from oracle import nnv_oracle as o
    for i in range(count):
        exp = o.star_from_box(lbs[:, i], ubs[:, i]).V
        assert np.array_equal(sets[i].V, exp)
        rows = rs.randint(0, N, size=min(N, 9))
        assert np.array_equal(sets[i]._h.fetch_rows(rows), exp[rows])
    assert ctx.pool_stats()[0] == before
