"""What boxes and released arrays hold on to: a box array that could never be written whole is refused where it is made,
staging memory stays bounded whatever the array's size, and the queue of released arrays stays bounded in a loop."""
import ctypes as C

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
