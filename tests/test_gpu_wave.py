"""The wave-per-task extension kernel against the oracle, at the sizes where it
can go wrong: query lengths around its widths of 64*C columns, bands around the
width of each frame (2w + 1 + C columns), frames that travel past their base
windows of 256, first rows that reach past the frame, and N bases.  The batch
sizes are those around which one launch takes all tasks, two launches take them
beside each other, and the bins take them."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_pair import FIELDS, SCORINGS, make_tasks, repeat

pytestmark = pytest.mark.gpu

DIRECT_MAX = 98304

CASES = {
    "widths": dict(qlens=(193, 224, 225, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048), n=140,
                   h0=lambda r, q: r.integers(1, 300), w=(3000,)),
    "frames": dict(qlens=(257, 300, 513, 700, 1025, 1500, 2048), n=210, h0=lambda r, q: r.integers(20, 200),
                   w=(125, 126, 251, 252, 503, 504, 1007, 1008), sub=0.02),
    "thin": dict(qlens=(257, 400, 900, 2048), n=160, h0=lambda r, q: r.integers(20, 200), w=(0, 1, 2, 3, 5, 20, 64),
                 sub=0.02),
    "first_row": dict(qlens=(260, 512, 800, 1300, 2000), n=150, h0=lambda r, q: r.integers(200, 4000),
                      w=(10, 100, 125, 250, 300), sub=0.1),
    "n_bases": dict(qlens=(200, 300, 600, 1100, 2048), n=100, h0=lambda r, q: r.integers(20, 300), w=(50, 100, 200, 400),
                    n_frac=0.02),
    "long_targets": dict(qlens=(230, 256, 258, 1000), n=80, h0=lambda r, q: r.integers(500, 3000), w=(100, 2000),
                         tail=(255, 256, 257, 600)),
    "narrow": dict(qlens=(1, 2, 31, 63, 64, 65, 100, 127, 128, 129, 150, 192), n=240, h0=lambda r, q: r.integers(1, 300),
                   w=(0, 1, 5, 20, 30, 31, 32, 62, 63, 100), n_frac=0.01),
    "no_target": dict(qlens=(200, 300, 600, 1100, 2048), n=20, h0=lambda r, q: r.integers(1, 60), w=(100,), tlen=0),
}


@pytest.mark.parametrize("scoring", sorted(SCORINGS))
@pytest.mark.parametrize("case", sorted(CASES))
def test_wave_kernel_equals_the_oracle(engine, case, scoring):
    from bsbolt_amd.bsx import Scoring
    kw = dict(CASES[case])
    t = make_tasks(100 + sorted(CASES).index(case), list(kw.pop("qlens")), kw.pop("n"), kw.pop("h0"), kw.pop("w"), **kw)
    sc = Scoring.make(**SCORINGS[scoring])
    want, _ = O.extend2_batch(t, nthreads=8, scoring=sc.as_dict())
    for n in (len(t), 2049, DIRECT_MAX, DIRECT_MAX + 1) if scoring == "asym" else (len(t), 2049):
        b, idx = repeat(t, n)
        got = engine.extend(b, sc)
        for k in FIELDS:
            assert np.array_equal(got[k], want[k][idx]), f"{k}, {n} tasks"


@pytest.mark.parametrize("n", (1, 7, 2048, 2049, 5000))
def test_unbinned_batches_reject_like_the_bins(engine, n):
    from bsbolt_amd.bsx import BsxError
    t = make_tasks(7, (20, 100, 200, 300), n, lambda r, q: r.integers(1, 100), (100, 200))
    want, _ = O.extend2_batch(t, nthreads=8)
    bad = np.unique(np.linspace(0, n - 1, min(n, 9)).astype(int))
    t.h0[bad[::2]] = 0
    t.qlen[bad[1::2]] = 0
    out = {k: np.full(n, -12345, np.int32) for k in FIELDS[:6]}
    with pytest.raises(BsxError, match=rf"{len(bad)} task\(s\) rejected.*first is task 0"):
        engine.extend(t, out=out, cells=False)
    good = np.ones(n, bool)
    good[bad] = False
    for k in FIELDS[:6]:
        assert (out[k][bad] == -12345).all() and np.array_equal(out[k][good], want[k][good]), k


@pytest.mark.parametrize("cls", (0, 1, 2, 3))
@pytest.mark.parametrize("scoring", ("asym", "bsbolt", "gap25"))
def test_frames_of_small_batches_fail_as_the_frame_kernels_do(cls, scoring):
    """The same results and the same count of failed frames as the frame kernels,
    which a timed call still runs."""
    from bsbolt_amd import bsx
    from bsbolt_amd.bsx import Scoring
    sc = Scoring.make(**SCORINGS[scoring])
    parts = [make_tasks(31, (5, 24, 25, 40, 41, 80, 81, 100, 144, 145, 150, 224), 1800, lambda r, q: r.integers(1, 150),
                        (0, 3, 10, 12, 20, 40, 100), sub=0.05),
             make_tasks(32, (30, 60, 120, 250), 400, lambda r, q: r.integers(100, 900), (5, 30, 100), sub=0.1),
             make_tasks(33, (30, 90, 200, 500), 200, lambda r, q: r.integers(1, 200), (100,), n_frac=0.02)]
    e = bsx.Engine(0)
    try:
        e.set_band_policy(bsx.BAND_FIXED, cls)
        for t in parts:
            want, _ = O.extend2_batch(t, nthreads=8, scoring=sc.as_dict())
            seen = []
            for n, timed in ((len(t), 0), (len(t), 1), (5000, 0), (5000, 1)):
                b, idx = repeat(t, n)
                e.set_kernel_timing(timed)
                got = e.extend(b, sc)
                for k in FIELDS:
                    assert np.array_equal(got[k], want[k][idx]), (k, n, timed)
                seen.append(np.asarray(e.band_stats()).tolist())
            assert seen[0] == seen[1] and seen[2] == seen[3], cls
    finally:
        e.close()
