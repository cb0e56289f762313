"""The slots of bsx_kernel_times: bsx_ext_bin_limits' bins are the plain kernels,
the four frame classes follow them and the predictor is slot 15.  Every plain
kernel has its time in one of them."""
import numpy as np
import pytest

from bsbolt_amd import bsx
from test_gpu_pair import make_tasks, repeat


def test_classes_follow_the_plain_bins():
    lim = bsx.ext_bin_limits()
    assert len(lim) == len(bsx.EXT_SHAPES) == 11
    assert len(lim) + bsx.BAND_CLASSES - 1 == bsx.TIMED_SLOTS - 1
    assert (np.diff(lim[:bsx.EXT_QUERY_BINS]) > 0).all()
    assert (np.diff(lim[bsx.EXT_QUERY_BINS:]) > 0).all()


# One kind of task per batch; below 65,536 tasks none runs the pair kernels.
@pytest.mark.gpu
@pytest.mark.parametrize("qlen,n,slot", [(20, 4000, 9), (64, 4000, 9), (96, 4000, 9), (97, 4000, 10), (128, 4000, 10),
                                         (129, 4000, 10), (192, 4000, 10), (200, 4000, 5), (500, 4000, 5),
                                         (32, 65536, 0), (96, 65536, 2)])
def test_every_plain_kernel_is_timed(qlen, n, slot):
    e = bsx.Engine(0)
    try:
        e.set_side_streams(False)  # each kernel by itself
        b, _ = repeat(make_tasks(5, (qlen,), 200, lambda r, q: r.integers(20, 50), (100,), sub=0.02), n)
        for _ in range(2):  # a kernel's first launch loads it
            e.set_kernel_timing(1)
            e.extend(b)
            ms, calls = e.kernel_times()
        assert calls == 1 and int(np.argmax(ms)) == slot and (ms[11:] == 0).all(), ms
        e.set_band_policy(bsx.BAND_FIXED, 2)
        e.set_kernel_timing(1)
        e.extend(b)
        ms, calls = e.kernel_times()
        assert calls == 1 and [s for s in range(11, 16) if ms[s] > 0] == [13], ms
    finally:
        e.close()
