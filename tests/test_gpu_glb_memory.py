"""A CIGAR batch large enough for the two-tasks-per-lane kernels on a GPU without
memory left for their scratch: the group kernels take it, in an eager call and in
a graph captured then."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_gpair import PAIR_MIN, make_tasks, repeat

pytestmark = pytest.mark.gpu
GIB = 1 << 30


def _free_bytes():
    path = next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x)
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert C.CDLL(path).hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_large_cigar_batch_without_room_for_the_pair_scratch():
    from bsbolt_amd import bsx
    t = make_tasks(3, 400, (70, 150), (3, 8, 15, 31))
    slot = 64
    os_, on, oc, _ = O.global2_batch(t, slot, nthreads=8)
    oc = np.where(np.arange(slot)[None, :] < np.maximum(on, 0)[:, None], oc, 0)
    b, idx = repeat(t, PAIR_MIN + 5)
    e = bsx.Engine(0)
    held = []
    try:
        dev = {f: e.to_device(getattr(b, f)) for f in ("query", "q_off", "qlen", "target", "t_off", "tlen", "w")}
        outs = {"score": e.empty((len(b),), np.int32), "n_cigar": e.empty((len(b),), np.int32),
                "cigar": e.empty((len(b) * slot,), np.uint32)}
        ptrs = {f: v.ptr for f, v in {**dev, **outs}.items()}
        ptrs.update(n=PAIR_MIN - 1, cigar_slot=slot)
        e.set_global_zslot(16384)  # scratch of 0.8 GB a workspace on 256 CUs
        e.global_device(ptrs)      # the context's own is there
        e.sync()
        ptrs["n"] = len(b)
        keep = 7 * GIB // 4        # what a graph's workspace takes, but not the pair scratch (2.5 GiB)
        while _free_bytes() - keep > GIB // 8:
            held.append(e.L.bsx_dev_alloc(e.ctx, min(16 * GIB, _free_bytes() - keep)))
            assert held[-1], e.last_error()
        print(f"{len(held)} blocks held, {_free_bytes() / GIB:.2f} GiB free", flush=True)

        def check():
            n = outs["n_cigar"].numpy()
            assert np.array_equal(outs["score"].numpy(), os_[idx]) and np.array_equal(n, on[idx])
            cg = outs["cigar"].numpy().reshape(len(b), slot)
            assert np.array_equal(np.where(np.arange(slot)[None, :] < np.maximum(n, 0)[:, None], cg, 0), oc[idx])

        e.global_device(ptrs)
        e.sync()
        check()
        g = e.capture_global(ptrs)
        try:
            for _ in range(3):
                e.L.bsx_memcpy(e.ctx, outs["score"].ptr, np.zeros(len(b), np.int32).ctypes.data, 4 * len(b), 1)
                g.launch()
                e.sync()
                check()
        finally:
            g.close()
        for p in held:
            e.L.bsx_dev_free(e.ctx, p)
        held.clear()
        e.global_device(ptrs)  # with room again
        e.sync()
        check()
    finally:
        for p in held:
            e.L.bsx_dev_free(e.ctx, p)
        e.close()
