"""The two-tasks-per-lane extension kernel against the oracle, at the sizes
where it can go wrong: query lengths around its eight-column blocks and bins,
scores, targets and gap costs at the limits of its range, bands whose first row
reaches past them, and batches around the size from which it runs."""
import numpy as np
import pytest

from bsbolt_amd.tasks import ExtTasks
from oracle import oracle as O

pytestmark = pytest.mark.gpu
FIELDS = ("score", "qle", "tle", "gtle", "gscore", "max_off", "cells")
PAIR_MIN = 98305


def make_tasks(seed, qlens, n, h0, w, eb=(0, 5, 30), tail=(0, 1, 40), sub=0.03, n_frac=0.0, tlen=None):
    """n tasks with query lengths from `qlens`: targets follow the query with
    substitutions and a short indel in a third of them, half of them unrelated
    after the first few bases, then `tail` more bases (or a fixed `tlen`)."""
    rng = np.random.default_rng(seed)
    pairs, h0s, ws, ebs = [], [], [], []
    for k in range(n):
        ql = int(qlens[k % len(qlens)])
        q = rng.integers(0, 4, ql).astype(np.uint8)
        t = np.where(rng.random(ql) < sub, rng.integers(0, 4, ql), q).astype(np.uint8)
        if rng.random() < 0.33 and ql > 4:
            p, g = int(rng.integers(1, ql)), int(rng.integers(1, 5))
            t = np.concatenate([t[:p], rng.integers(0, 4, g), t[p:]]) if rng.random() < 0.5 else np.delete(t, slice(p, p + g))
        if rng.random() < 0.5:
            keep = int(rng.integers(0, len(t) + 1))
            t[keep:] = rng.integers(0, 4, len(t) - keep)
        m = int(rng.choice(tail)) if tlen is None else max(0, tlen - len(t))
        t = np.concatenate([t, rng.integers(0, 4, m)]).astype(np.uint8)[:tlen]
        if n_frac:
            q[rng.random(ql) < n_frac] = 4
            t[rng.random(len(t)) < n_frac] = 4
        pairs.append((q, t))
        h0s.append(int(h0(rng, ql)))
        ws.append(int(rng.choice(w)))
        ebs.append(int(rng.choice(eb)))
    return ExtTasks.from_pairs(pairs, h0s, ws, ebs)


def repeat(t, n):
    idx = np.arange(n) % len(t)
    return ExtTasks(t.query, t.q_off[idx], t.qlen[idx], t.target, t.t_off[idx], t.tlen[idx], t.h0[idx], t.w[idx],
                    t.end_bonus[idx]), idx


CASES = {
    # every query length of the bins up to 128 bases, h0 as seeds give it
    "lengths": dict(qlens=range(1, 130), n=1935, h0=lambda r, q: r.integers(1, 140), w=(100,)),
    "long_lengths": dict(qlens=(127, 128, 129, 135, 136, 137, 160, 191, 200, 222, 223, 224, 225, 230), n=700,
                         h0=lambda r, q: r.integers(1, max(2, 256 - q)), w=(100, 300)),
    # bands narrower than the query: the cap cuts columns, the first row may reach past the band
    "bands": dict(qlens=(1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 95, 96), n=1200, h0=lambda r, q: r.integers(1, 60),
                  w=(0, 1, 2, 7, 16, 40)),
    # the first row's values reach far past the band, and the band comes back to them
    "first_row": dict(qlens=(40, 64, 96, 100, 128), n=1500, h0=lambda r, q: r.integers(60, 380), w=(1, 3, 10, 30, 60),
                      sub=0.15),
    "first_row_long": dict(qlens=(129, 150, 180, 224), n=600, h0=lambda r, q: r.integers(20, 256 - q + 1),
                           w=(1, 3, 10, 30, 60, 100), sub=0.1),
    # N bases in query and target
    "n_bases": dict(qlens=(5, 24, 40, 64, 90, 96), n=600, h0=lambda r, q: r.integers(1, 80), w=(100,), n_frac=0.03),
    # scores at and past the kernel's limit (h0 + qlen = 511 runs in it, 512 does not)
    "scores": dict(qlens=(1, 16, 32, 64, 96), n=600, h0=lambda r, q: 511 - q + r.integers(-1, 2), w=(100, 500),
                   sub=0.0),
    "scores_long": dict(qlens=(128, 129, 200, 224), n=400, h0=lambda r, q: (511 if q <= 128 else 255) - q + r.integers(-1, 2),
                        w=(100, 500), sub=0.0),
    # target lengths at and past its limit, and empty targets
    "targets": dict(qlens=(1, 32, 64, 96, 128), n=300, h0=lambda r, q: 511 - q, w=(700,), tail=(0,), tlen=640),
    "long_targets": dict(qlens=(1, 32, 64, 96), n=300, h0=lambda r, q: 511 - q, w=(700,), tail=(0,), tlen=641),
    "no_target": dict(qlens=(1, 32, 96, 128, 200), n=60, h0=lambda r, q: r.integers(1, 60), w=(100,), tlen=0),
}
SCORINGS = {
    "bsbolt": dict(),
    "asym": dict(o_del=4, e_del=2, o_ins=7, e_ins=1, zdrop=30, a=2, b=5),
    "gap25": dict(o_del=0, e_del=25, o_ins=3, e_ins=25, zdrop=0),
    "no_zdrop_25": dict(o_del=5, e_del=25, o_ins=2, e_ins=24, zdrop=30000),
    "gap26": dict(o_del=0, e_del=26, o_ins=3, e_ins=2, zdrop=20000),
}


@pytest.mark.parametrize("scoring", sorted(SCORINGS))
@pytest.mark.parametrize("case", sorted(CASES))
def test_pair_kernel_equals_the_oracle(engine, case, scoring):
    from bsbolt_amd.bsx import Scoring
    kw = dict(CASES[case])
    t = make_tasks(sorted(CASES).index(case), list(kw.pop("qlens")), kw.pop("n"), kw.pop("h0"), kw.pop("w"), **kw)
    sc = Scoring.make(**SCORINGS[scoring])
    want, _ = O.extend2_batch(t, nthreads=8, scoring=sc.as_dict())
    for n in (PAIR_MIN - 1, PAIR_MIN + 77):
        b, idx = repeat(t, n)
        got = engine.extend(b, sc)
        for k in FIELDS:
            assert np.array_equal(got[k], want[k][idx]), f"{k}, {n} tasks"
