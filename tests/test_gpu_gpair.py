"""The two-tasks-per-lane CIGAR kernel against the oracle: every band width of
its bins, tasks at the limits of its range, and batches around the size from
which it runs."""
import numpy as np
import pytest

from bsbolt_amd.tasks import GlbTasks
from oracle import oracle as O

pytestmark = pytest.mark.gpu
PAIR_MIN = 131072


def make_tasks(seed, n, qlens, bands, sub=0.05, gap=0.5, n_frac=0.0):
    """n tasks: the target is the query with substitutions and, in a share
    `gap` of them, an insertion or deletion that the band can hold."""
    rng = np.random.default_rng(seed)
    pairs, ws = [], []
    for k in range(n):
        ql, w = int(qlens[k % len(qlens)]), int(bands[(k // len(qlens)) % len(bands)])
        q = rng.integers(0, 4, ql).astype(np.uint8)
        t = np.where(rng.random(ql) < sub, rng.integers(0, 4, ql), q).astype(np.uint8)
        if rng.random() < gap and w > 0:
            g = int(rng.integers(1, w + 1))
            p = int(rng.integers(0, ql + 1))
            if rng.random() < 0.5:
                t = np.concatenate([t[:p], rng.integers(0, 4, g).astype(np.uint8), t[p:]])
            elif ql > g:
                p = min(p, ql - g)
                t = np.delete(t, slice(p, p + g))
        if n_frac:
            q[rng.random(ql) < n_frac] = 4
            t[rng.random(len(t)) < n_frac] = 4
        pairs.append((q, t))
        ws.append(max(w, abs(len(t) - ql)))
    return GlbTasks.from_pairs(pairs, ws)


def repeat(t, n):
    idx = np.arange(n) % len(t)
    return GlbTasks(t.query, t.q_off[idx], t.qlen[idx], t.target, t.t_off[idx], t.tlen[idx], t.w[idx]), idx


CASES = {
    # every band width the bins take, and the first one past them
    "bands": dict(n=900, qlens=(33, 70, 150), bands=range(0, 33)),
    # queries shorter than the band, single bases
    "short": dict(n=600, qlens=(1, 2, 3, 7, 8, 9, 20), bands=(0, 1, 3, 7, 8, 15, 31)),
    # target lengths around the limit of 320 and the row steps
    "rows": dict(n=300, qlens=(9, 10, 11, 310, 318, 320, 321, 330), bands=(3, 9, 12)),
    "n_bases": dict(n=300, qlens=(40, 150, 250), bands=(4, 9, 20), n_frac=0.03),
    "unrelated": dict(n=400, qlens=(60, 150), bands=(3, 8, 11, 16, 25), sub=0.9),
}
SCORINGS = {
    "bsbolt": dict(),
    "asym": dict(o_del=4, e_del=2, o_ins=7, e_ins=1, a=2, b=5),
    "free_open": dict(o_del=0, e_del=1, o_ins=0, e_ins=3),
    # scores of the longer tasks leave the kernel's 16 bits
    "large": dict(o_del=30, e_del=40, o_ins=20, e_ins=50, a=20, b=60),
}


@pytest.mark.parametrize("scoring", sorted(SCORINGS))
@pytest.mark.parametrize("case", sorted(CASES))
def test_pair_kernel_equals_the_oracle(engine, case, scoring):
    from bsbolt_amd.bsx import Scoring
    kw = dict(CASES[case])
    t = make_tasks(sorted(CASES).index(case), kw.pop("n"), list(kw.pop("qlens")), list(kw.pop("bands")), **kw)
    sc = Scoring.make(**SCORINGS[scoring])
    slot = 64
    os_, on, oc, _ = O.global2_batch(t, slot, nthreads=8, scoring=sc.as_dict())
    # a CIGAR of more than `slot` words is reported, not compared
    for n in (PAIR_MIN - 1, PAIR_MIN + 77):
        b, idx = repeat(t, n)
        (s, nc, cg), rc = engine.global_(b, sc, slot=slot, raise_on_error=False)
        assert np.array_equal(s, os_[idx])
        fits = on[idx] >= 0
        assert np.array_equal(nc[fits], on[idx][fits]) and (nc[~fits] == -1).all()
        used = (np.arange(slot)[None, :] < np.maximum(on, 0)[:, None])
        assert np.array_equal(np.where(used[idx], cg, 0), np.where(used, oc, 0)[idx])


def test_scores_without_cigars(engine):
    t = make_tasks(9, 500, (30, 100, 150), range(3, 32))
    os_, _, _, _ = O.global2_batch(t, 320, nthreads=8)
    b, idx = repeat(t, PAIR_MIN + 5)
    s, nc, _ = engine.global_(b, cigar=False)
    assert np.array_equal(s, os_[idx]) and (nc == 0).all()
