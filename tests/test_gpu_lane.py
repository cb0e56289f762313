"""The task-per-lane extension kernel, which takes the queries of up to 64 bases
outside the pair kernels' range, against the oracle at the sizes where it can go
wrong: query lengths around its widths, scores and targets from the range's limits
up to those of long reads, targets around its 16-base windows, empty targets, gap
costs the pair kernels do not take, and lists that end inside a wave."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_pair import FIELDS, make_tasks, repeat

pytestmark = pytest.mark.gpu

LENGTHS = (1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65)
CASES = {
    "scores": dict(n=850, h0=lambda r, q: 512 - q + r.integers(0, 3), w=(100, 500), sub=0.0),
    "long_reads": dict(n=850, h0=lambda r, q: r.integers(512, 4000), w=(0, 1, 2, 7, 30, 100), sub=0.05),
    "windows": dict(n=850, h0=lambda r, q: r.integers(600, 900), w=(20, 100), tail=(0, 1, 15, 16, 17, 31, 33, 64)),
    "long_targets": dict(n=170, h0=lambda r, q: r.integers(1, 900), w=(700,), tail=(0,), tlen=641),
    "n_bases": dict(n=850, h0=lambda r, q: r.integers(600, 700), w=(100,), n_frac=0.03),
    "no_target": dict(n=68, h0=lambda r, q: r.integers(600, 700), w=(100,), tlen=0),
}
SCORINGS = {
    "bsbolt": dict(),
    "asym": dict(o_del=4, e_del=2, o_ins=7, e_ins=1, zdrop=30, a=2, b=5),
    "gap26": dict(o_del=0, e_del=26, o_ins=3, e_ins=26, zdrop=0),
}


@pytest.mark.parametrize("scoring", sorted(SCORINGS))
@pytest.mark.parametrize("case", sorted(CASES))
def test_lane_kernel_equals_the_oracle(engine, case, scoring):
    from bsbolt_amd.bsx import Scoring
    kw = dict(CASES[case])
    t = make_tasks(300 + sorted(CASES).index(case), LENGTHS, kw.pop("n"), kw.pop("h0"), kw.pop("w"), **kw)
    sc = Scoring.make(**SCORINGS[scoring])
    want, _ = O.extend2_batch(t, nthreads=8, scoring=sc.as_dict())
    for n in (98305, 98305 + 64 * 77 + 1):
        b, idx = repeat(t, n)
        got = engine.extend(b, sc)
        for k in FIELDS:
            assert np.array_equal(got[k], want[k][idx]), f"{k}, {n} tasks"


def test_short_rows_outside_the_pair_range_cost_less_than_group_rows():
    """A row of a query of up to 64 bases takes 43-59 ps of a full chip in the
    task-per-lane kernel and 109 in the 16x6 group kernel, which a query of 96
    bases runs; every task here runs all of its 100 rows."""
    from bsbolt_amd import bsx
    from bsbolt_amd.tasks import RESULT_FIELDS
    e = bsx.Engine(0)
    try:
        us = {}
        for q in (32, 64, 96):
            t = make_tasks(9, (q,), 2000, lambda r, _: 2000, (200,), sub=0.0, tlen=100)
            b, _ = repeat(t, 600_000)
            keep, ptrs = e.tasks_to_device(b)
            outs = {k: e.empty((len(b),), np.int32) for k in RESULT_FIELDS}
            ptrs.update({k: v.ptr for k, v in outs.items()}, n=len(b))
            sc = bsx.Scoring.make(zdrop=0)
            best = 1e9
            for _ in range(5):
                e.timer_start()
                e.extend_device(ptrs, sc)
                best = min(best, e.timer_stop())
            e.sync()
            us[q] = best * 1e3
            del keep, outs
        print(f"us per call by query length: {us}", flush=True)
        assert us[32] < 0.75 * us[96] and us[64] < 0.75 * us[96], us
    finally:
        e.close()
