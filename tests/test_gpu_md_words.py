"""The NM / MD:Z / XB:Z kernel against the oracle where its walk by words of 32
bases can go wrong: op lengths around a word, reads around 32 bases, N bases,
numbers of three and four digits, windows at the ends of the reference, CIGARs
that leave them, and slots that overflow or do not start on a dword."""
import numpy as np
import pytest

import md_cases as M
from oracle import oracle as O
from test_gpu_md import _run, eng  # noqa: F401

pytestmark = pytest.mark.gpu
GLEN = 4000


def make(seed, n, lens, ops, p_n=0.0, p_err=0.02, over=0.0):
    """n random regions with CIGARs of `ops` ops; M lengths from `lens`."""
    g, pac, opac, l_pac, crick_l = M.index(GLEN, 9)
    rng = np.random.default_rng(seed)
    rbs, res, oqs, cgs = [], [], [], []
    for k in range(n):
        cg = []
        for x in range(int(rng.choice(ops))):
            cg.append((int(rng.choice(lens)), 0) if x % 2 == 0 else (int(rng.integers(1, 40)), int(rng.integers(1, 3))))
        if rng.random() < 0.1:
            cg.insert(0, (3, 2))
        rlen = max(1, sum(c for c, op in cg if op != 1))
        q, edge = int(rng.integers(4)), rng.random()
        lo = 0 if edge < 0.1 else GLEN - rlen if edge < 0.2 else int(rng.integers(0, GLEN - rlen + 1))
        rb = q * GLEN + lo
        re = rb + (rlen if rng.random() >= over else max(1, rlen - int(rng.integers(1, 6))))
        w = O.get_seq(l_pac, opac, rb, rb + rlen).astype(np.uint8)
        w = w if rb < l_pac else w[::-1]
        crick = (crick_l <= rb < l_pac) or rb >= crick_l + l_pac
        parts, y = [], 0
        for c, op in cg:
            if op == 0:
                parts.append(w[y:y + c])
            if op == 1:
                parts.append(rng.integers(0, 4, c).astype(np.uint8))
            y += c if op != 1 else 0
        o = np.concatenate(parts + [rng.integers(0, 4, int(rng.integers(0, 3))).astype(np.uint8)])
        ref, conv = (2, 0) if crick else (1, 3)
        o = np.where((o == ref) & (rng.random(len(o)) < rng.random()), conv, o)
        o = np.where(rng.random(len(o)) < p_err, rng.integers(0, 4, len(o)), o)
        o = np.where(rng.random(len(o)) < p_n, 4, o).astype(np.uint8)
        rbs.append(rb), res.append(re), oqs.append(o if rb < l_pac else o[::-1])
        cgs.append(np.array([c << 4 | op for c, op in cg], np.uint32))
    return (opac, l_pac, crick_l, rbs, res, oqs, cgs)


CASES = {
    "words": dict(n=600, lens=(1, 2, 31, 32, 33, 63, 64, 65, 100, 150), ops=(1, 2, 3, 5)),
    "short": dict(n=400, lens=(1, 3, 10, 28, 30), ops=(1, 3)),
    "n_bases": dict(n=300, lens=(20, 90, 150), ops=(1, 3), p_n=0.03),
    "far": dict(n=60, lens=(90, 110, 999, 1000, 1001, 1300), ops=(1, 3), p_err=0.0003),
    "noise": dict(n=200, lens=(40, 150), ops=(1, 3), p_err=0.9),
    "past_the_window": dict(n=300, lens=(30, 64, 150), ops=(1, 3), over=0.5),
}


@pytest.mark.parametrize("slots", ((None, None), (40, 64), (61, 47)))
@pytest.mark.parametrize("case", sorted(CASES))
def test_md_by_words_equals_the_oracle(eng, case, slots):  # noqa: F811
    t = make(sorted(CASES).index(case), **CASES[case])
    kw = {} if slots[0] is None else dict(md_slot=slots[0], xb_slot=slots[1])
    got = _run(eng, *t, **kw)
    opac, l_pac, crick_l, rbs, res, oqs, cgs = t
    for i in range(len(rbs)):
        st, md, xb, nm, meth = O.gen_md(l_pac, opac, rbs[i], res[i], crick_l, oqs[i], cgs[i])
        if slots[0] is not None and st == 0 and (len(md) > slots[0] or len(xb) > slots[1]):
            st, md, xb, nm, meth = -1, "", "", -1, [0, 0, 0, 0]
        if slots[0] is not None and st < 0 and got["status"][i] in (-1, -2):
            st = got["status"][i]  # the first of the two; which one it is is not compared
        assert got["status"][i] == st, i
        if st == 0:
            assert (got["md"][i], got["xb"][i], int(got["nm"][i]), list(got["meth"][i])) == (md, xb, nm, meth), i
        else:
            assert got["md"][i] == "" and got["xb"][i] == "" and got["nm"][i] == -1, i
