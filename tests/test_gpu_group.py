"""The group extension kernels (16-32 lanes a task), which take the queries of
65-192 bases outside the pair kernels' range in large batches: against the oracle
with every group shape and chunk size of the tuning table, in lists that fit one
chunk a block and in lists of many; and the even use of the chip by a list whose
runs differ in length."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_pair import FIELDS, make_tasks, repeat

pytestmark = pytest.mark.gpu

CASES = {
    "lengths": dict(qlens=(65, 66, 95, 96, 97, 98, 127, 128, 129, 130, 160, 191, 192), h0=lambda r, q: r.integers(512, 900),
                    w=(3, 30, 100, 200), sub=0.05),
    "first_bin": dict(qlens=(65, 80, 96), h0=lambda r, q: r.integers(512, 600), w=(100,), n_frac=0.02),
    "long_targets": dict(qlens=(70, 100, 150), h0=lambda r, q: r.integers(1, 900), w=(700,), tail=(0,), tlen=641),
}


@pytest.mark.parametrize("table", [None, [16, 16, 1, 0], [64, 32, 0, 1], [128, 64, 1, 1]], ids=str)
@pytest.mark.parametrize("case", sorted(CASES))
def test_group_kernels_equal_the_oracle(engine, case, table):
    from bsbolt_amd.bsx import Scoring
    kw = dict(CASES[case])
    t = make_tasks(400 + sorted(CASES).index(case), kw.pop("qlens"), 260, kw.pop("h0"), kw.pop("w"), **kw)
    old = engine.get_tuning()[0]
    try:
        engine.set_tuning(table)
        for scoring, n in ((dict(), 98305), (dict(o_del=4, e_del=2, o_ins=7, e_ins=1, zdrop=30, a=2, b=5), 98305),
                           (dict(), 300_007), (dict(o_del=0, e_del=26, o_ins=3, e_ins=26, zdrop=0), 300_007)):
            sc = Scoring.make(**scoring)
            want, _ = O.extend2_batch(t, nthreads=8, scoring=sc.as_dict())
            b, idx = repeat(t, n)
            got = engine.extend(b, sc)
            for k in FIELDS:
                assert np.array_equal(got[k], want[k][idx]), f"{k}, {n} tasks, {scoring}"
    finally:
        engine.set_tuning(old)


def test_long_runs_spread_over_the_chip():
    """600,000 tasks that run all of their rows, 34-35 on average: alike, or a
    twentieth of them 300 rows and the others 20.  The lists are longest first, so
    fixed shares of them leave all the long runs to a few blocks."""
    from bsbolt_amd import bsx
    from bsbolt_amd.tasks import RESULT_FIELDS, ExtTasks
    e = bsx.Engine(0)
    try:
        us = {}
        for name, tlens in (("alike", (35,)), ("mixed", (300,) + (20,) * 19)):
            parts = [make_tasks(9, (96,), 100, lambda r, _: 2000, (200,), sub=0.0, tlen=x) for x in tlens]
            pairs = [(p.query_of(i), p.target_of(i)) for i in range(100) for p in parts]
            b, _ = repeat(ExtTasks.from_pairs(pairs, [2000] * len(pairs), [200] * len(pairs), [5] * len(pairs)), 600_000)
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
            us[name] = best * 1e3
            del keep, outs
        print(f"us per call: {us}", flush=True)
        assert us["mixed"] < 1.6 * us["alike"], us
    finally:
        e.close()
