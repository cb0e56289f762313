"""The NM / MD:Z / XB:Z kernel with a reference that starts at any byte of a dword:
the same results, by the walk of 32 bases at a time."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_md import _pack_cigars
from test_gpu_md_words import CASES, GLEN, make

pytestmark = pytest.mark.gpu


def device(e, t, off, reps=1):
    """The regions of `t` on the device, `reps` times; opac at byte `off` of a dword."""
    opac, l_pac, crick_l, rbs, res, oqs, cgs = t
    cig, nc = _pack_cigars(cgs)
    oq_off = np.concatenate([[0], np.cumsum([len(x) for x in oqs])[:-1]]).astype(np.uint64)
    ql = np.array([len(x) for x in oqs], np.int32)
    n = len(rbs) * reps
    host = {"rb": np.asarray(rbs, np.int64), "re": np.asarray(res, np.int64), "oq_off": oq_off, "l_query": ql,
            "n_cigar": nc, "cigar": cig}
    keep = {k: e.to_device(np.ascontiguousarray(np.tile(v, (reps,) + (1,) * (v.ndim - 1)))) for k, v in host.items()}
    keep["oquery"] = e.to_device(np.concatenate(oqs).astype(np.uint8))
    keep["opac"] = e.to_device(np.concatenate([np.full(off, 0xa5, np.uint8), np.asarray(opac, np.uint8)]))
    ms, xs = int(4 * ql.max() + 4 * cig.shape[1] + 16), int(4 * ql.max() + 16)
    out = {"md": e.empty((n, ms), np.uint8), "xb": e.empty((n, xs), np.uint8), "meth": e.empty((n, 4), np.int32)}
    out.update({k: e.empty((n,), np.int32) for k in ("md_len", "xb_len", "nm", "status")})
    ptrs = {k: v.ptr for k, v in {**keep, **out}.items()}
    ptrs["opac"] += off
    ptrs.update(n=n, l_pac=int(l_pac), crick_l=int(crick_l), cigar_slot=int(cig.shape[1]), md_slot=ms, xb_slot=xs)
    return keep, out, ptrs


@pytest.mark.parametrize("off", (0, 1, 2, 3))
@pytest.mark.parametrize("case", ("words", "short", "past_the_window"))
def test_any_alignment_of_the_reference(case, off):
    from bsbolt_amd import bsx
    t = make(sorted(CASES).index(case), **CASES[case])
    opac, l_pac, crick_l, rbs, res, oqs, cgs = t
    e = bsx.Engine(0)
    try:
        keep, out, ptrs = device(e, t, off)
        e.md_device(ptrs)
        e.sync()
        h = {k: v.numpy() for k, v in out.items()}
        for i in range(len(rbs)):
            st, md, xb, nm, meth = O.gen_md(l_pac, opac, rbs[i], res[i], crick_l, oqs[i], cgs[i])
            assert h["status"][i] == st, i
            if st == 0:
                got = (bytes(h["md"][i, :h["md_len"][i]]).decode(), bytes(h["xb"][i, :h["xb_len"][i]]).decode(),
                       int(h["nm"][i]), list(h["meth"][i]))
                assert got == (md, xb, nm, meth), i
        del keep, out
    finally:
        e.close()


def test_an_odd_reference_costs_no_more():
    """Base by base a call takes six times as long and more."""
    from bsbolt_amd import bsx
    t = make(3, 500, (150,), (1,), p_err=0.01)
    mid = [i for i, rb in enumerate(t[3]) if 100 < rb % GLEN < GLEN - 400]  # regions at the ends are walked base by base
    t = t[:3] + tuple([x[i] for i in mid] for x in t[3:])
    e = bsx.Engine(0)
    try:
        us = {}
        for off in (0, 1, 3):
            keep, out, ptrs = device(e, t, off, 200)
            best = 1e9
            for _ in range(5):
                e.timer_start()
                e.md_device(ptrs)
                best = min(best, e.timer_stop())
            us[off] = best * 1e3
            del keep, out
        print(f"us per call by byte offset: {us}", flush=True)
        assert max(us[1], us[3]) < 2 * us[0], us
    finally:
        e.close()
