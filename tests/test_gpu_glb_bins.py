"""The group CIGAR kernels of mid-size batches, whose launches beside each other
divide the direction slots by their lists: against the oracle where a batch is of
one kind, of two kinds very unevenly, and of all, at sizes around the slots one
kind can use; and the cost of bands of 25-32 against that of the next narrower."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_gpair import make_tasks

pytestmark = pytest.mark.gpu

# half bandwidths of the bins of 16, 24, 32, 64, 128 and 256 columns
KINDS = {"16": (4, 7), "24": (8, 11), "32": (12, 15), "64": (16, 31), "128": (33, 63), "256": (64, 110)}


def batch(kinds, n, rest=None, few=0):
    """n tasks of `kinds` in turn, the first `few` of them of `rest` instead."""
    from bsbolt_amd.tasks import GlbTasks
    parts = [make_tasks(20 + i, 60, (150,) if k in ("128", "256") else (63, 70, 150), KINDS[k]) for i, k in
             enumerate(list(kinds) + ([rest] if rest else []))]
    pairs = [(p.query[int(p.q_off[i]):][:p.qlen[i]], p.target[int(p.t_off[i]):][:p.tlen[i]])
             for p in parts for i in range(len(p))]
    t = GlbTasks.from_pairs(pairs, np.concatenate([p.w for p in parts]))
    per, main = len(parts[0]), len(kinds) * len(parts[0])
    idx = np.arange(n) % main
    if rest:
        idx[:few] = main + np.arange(few) % per
    idx = np.random.default_rng(3).permutation(idx)
    return t, GlbTasks(t.query, t.q_off[idx], t.qlen[idx], t.target, t.t_off[idx], t.tlen[idx], t.w[idx]), idx


CASES = [((k,), n, None, 0) for k in KINDS for n in (20481, 28673, 49185, 131071)] + \
        [(("16",), 60001, "32", 1), (("32",), 60001, "64", 33), (("64",), 60001, "32", 31), (("256",), 30001, "24", 7),
         (("24", "32"), 70003, "128", 129), (tuple(KINDS), 20481, None, 0), (tuple(KINDS), 131071, None, 0)]


@pytest.mark.parametrize("kinds,n,rest,few", CASES)
def test_bins_equal_the_oracle(engine, kinds, n, rest, few):
    t, b, idx = batch(kinds, n, rest, few)
    slot = 64
    os_, on, oc, _ = O.global2_batch(t, slot, nthreads=8)
    assert (on >= 0).all()
    oc = np.where(np.arange(slot)[None, :] < on[:, None], oc, 0)
    for side in (True, False) if n == 20481 else (True,):
        engine.set_side_streams(side)
        try:
            s, nc, cg = engine.global_(b, slot=slot)
        finally:
            engine.set_side_streams(True)
        assert np.array_equal(s, os_[idx]) and np.array_equal(nc, on[idx])
        assert np.array_equal(np.where(np.arange(slot)[None, :] < nc[:, None], cg, 0), oc[idx])


def test_bands_of_25_to_32_have_lanes_of_their_own():
    """8 lanes of 4 columns hold such a band as 8 of 3 hold one of 17-24; in the
    shape of 33-64 columns half the lanes would idle."""
    from bsbolt_amd import bsx
    e = bsx.Engine(0)
    try:
        us = {}
        for k in ("24", "32"):
            _, b, _ = batch((k,), 131_000)
            fields = ("query", "q_off", "qlen", "target", "t_off", "tlen", "w")
            dev = {f: e.to_device(getattr(b, f)) for f in fields}
            outs = {"score": e.empty((len(b),), np.int32), "n_cigar": e.empty((len(b),), np.int32),
                    "cigar": e.empty((len(b) * 64,), np.uint32)}
            ptrs = {f: v.ptr for f, v in {**dev, **outs}.items()}
            ptrs.update(n=len(b), cigar_slot=64)
            best = 1e9
            for _ in range(5):
                e.timer_start()
                e.global_device(ptrs)
                best = min(best, e.timer_stop())
            e.sync()
            us[k] = best * 1e3
            del dev, outs
        print(f"us per call by columns: {us}", flush=True)
        assert us["32"] < 1.6 * us["24"], us
    finally:
        e.close()
