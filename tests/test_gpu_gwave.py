"""The wave-per-task CIGAR kernel against the oracle: bands around its widths of
64, 128 and 256 columns, targets around its blocks of 64 rows, frames that
travel past their windows of 256 bases, CIGARs around 64 words, slots too small
for its directions, and batches around the size up to which it runs."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_gpair import SCORINGS, make_tasks, repeat

pytestmark = pytest.mark.gpu
DIRECT_MAX = 20480

CASES = {
    "bands": dict(n=700, qlens=(33, 70, 150, 300), bands=(0, 1, 2, 15, 16, 30, 31, 32, 33, 62, 63, 64, 65, 125, 126, 127)),
    "wide": dict(n=60, qlens=(200, 260, 300), bands=(125, 126, 127, 128, 250, 255, 300, 511)),
    "short": dict(n=300, qlens=(1, 2, 3, 31, 32, 33, 63, 64, 65), bands=(0, 1, 3, 31, 32, 70)),
    "rows": dict(n=300, qlens=(62, 63, 64, 65, 127, 128, 129, 191, 192, 193, 256, 257, 330), bands=(3, 9, 20, 40)),
    "long": dict(n=40, qlens=(900, 1600, 2500), bands=(2, 10, 12)),
    "n_bases": dict(n=200, qlens=(40, 150, 250), bands=(4, 20, 40, 80), n_frac=0.03),
    "unrelated": dict(n=200, qlens=(60, 150, 400), bands=(8, 25, 40, 70), sub=0.9),
}


@pytest.mark.parametrize("zslot", (1 << 16, 4096))
@pytest.mark.parametrize("scoring", sorted(SCORINGS))
@pytest.mark.parametrize("case", sorted(CASES))
def test_wave_kernel_equals_the_oracle(engine, case, scoring, zslot):
    from bsbolt_amd.bsx import Scoring
    kw = dict(CASES[case])
    t = make_tasks(50 + sorted(CASES).index(case), kw.pop("n"), list(kw.pop("qlens")), list(kw.pop("bands")), **kw)
    sc = Scoring.make(**SCORINGS[scoring])
    slot = 600
    os_, on, oc, _ = O.global2_batch(t, slot, nthreads=8, scoring=sc.as_dict())
    used = np.arange(slot)[None, :] < np.maximum(on, 0)[:, None]
    oc = np.where(used, oc, 0)
    engine.set_global_zslot(zslot)
    try:
        for n in (len(t), DIRECT_MAX, DIRECT_MAX + 1) if scoring == "asym" and case in ("bands", "rows") else (len(t),):
            b, idx = repeat(t, n)
            (s, nc, cg), rc = engine.global_(b, sc, slot=slot, raise_on_error=False)
            assert np.array_equal(s, os_[idx])
            fits = on[idx] >= 0
            assert np.array_equal(nc[fits], on[idx][fits]) and (nc[~fits] == -1).all()
            assert np.array_equal(np.where(used[idx], cg, 0), oc[idx])
            assert np.array_equal(engine.global_(b, sc, cigar=False)[0], os_[idx])
    finally:
        engine.set_global_zslot(1 << 16)


def test_cigars_around_a_register_of_words(engine):
    """Exactly 1 to 130 words, into slots that hold them or lack one word."""
    from bsbolt_amd.bsx import Scoring
    from bsbolt_amd.tasks import GlbTasks
    rng = np.random.default_rng(1)
    sc = Scoring.make(a=2, b=8, o_del=1, o_ins=1)
    pairs = []
    for words in (1, 3, 31, 61, 63, 65, 67, 127, 129):
        q, t = [], []
        for x in range(words // 2 + 1):
            m = rng.integers(0, 4, 12).astype(np.uint8)
            g = np.array([(m[-1] + 1) % 4], np.uint8)
            q += [m] if x == words // 2 or x % 2 == 0 else [m, g]
            t += [m] if x == words // 2 or x % 2 else [m, g]
        pairs.append((np.concatenate(q), np.concatenate(t)))
    t = GlbTasks.from_pairs(pairs, [2] * len(pairs))
    os_, on, oc, _ = O.global2_batch(t, 200, nthreads=2, scoring=sc.as_dict())
    assert on.max() > 128 and (on > 60).sum() > 4
    for slot in sorted({1, *[int(x) for x in on], *[int(x) - 1 for x in on if x > 1]}):
        (s, nc, cg), rc = engine.global_(t, sc, slot=slot, raise_on_error=False)
        assert np.array_equal(s, os_) and np.array_equal(nc, np.where(on <= slot, on, -1))
        for i in np.flatnonzero(on <= slot):
            assert np.array_equal(cg[i, :on[i]], oc[i, :on[i]]), (slot, i)
