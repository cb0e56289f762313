"""Host-memory batches where their arrays change route: gathered, copied from
where they lie or read in place, and CIGARs gathered or copied slot by slot."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_gpair import repeat as glb_repeat
from test_gpu_pair import FIELDS, make_tasks, repeat

pytestmark = pytest.mark.gpu


# 8 * 32768 bytes of offsets are the largest array gathered; 60 to 260 tasks lie
# around the largest batch read in place
@pytest.mark.parametrize("n", (1, 60, 100, 180, 260, 32768, 32769, 131072 + 98304))
def test_extension_batches_of_every_route(engine, n):
    t = make_tasks(3, (20, 60, 100), min(n, 400), lambda r, q: r.integers(1, 100), (100,))
    want, _ = O.extend2_batch(t, nthreads=8)
    b, idx = repeat(t, n)
    got = engine.extend(b)
    for k in FIELDS:
        assert np.array_equal(got[k], want[k][idx]), k


# CIGARs of up to `ops` words: a batch's room is 16 a task; more than 4,096 stay in their slots
@pytest.mark.parametrize("n,ops", ((1, 3), (1, 40), (5, 40), (300, 40), (300, 3), (65536, 3), (65540, 3), (2, 4200)))
def test_cigars_past_the_gathered_room(engine, n, ops):
    from bsbolt_amd.tasks import GlbTasks
    rng = np.random.default_rng(ops)
    pairs, ws = [], []
    for k in range(min(n, 50)):
        parts_q, parts_t = [], []
        for x in range(ops // 2):  # matches of 12 bases around gaps of one
            m = rng.integers(0, 4, 12).astype(np.uint8)
            g = np.array([(m[-1] + 1) % 4], np.uint8)
            parts_q += [m, g] if x % 2 else [m]
            parts_t += [m] if x % 2 else [m, g]
        pairs.append((np.concatenate(parts_q), np.concatenate(parts_t)))
        ws.append(2)
    t = GlbTasks.from_pairs(pairs, ws)
    from bsbolt_amd.bsx import Scoring
    sc = Scoring.make(a=2, b=8, o_del=1, o_ins=1)
    slot = ops + 8
    os_, on, oc, _ = O.global2_batch(t, slot, nthreads=8, scoring=sc.as_dict())
    b, idx = glb_repeat(t, n)
    b.w[-1:] = -1  # the last task is rejected
    (s, nc, cg), rc = engine.global_(b, sc, slot=slot, raise_on_error=False)
    good = np.arange(n) < n - 1
    assert np.array_equal(s[good], os_[idx][good]) and np.array_equal(nc[good], on[idx][good])
    assert ops == 3 or on.max() > 16
    used = np.arange(slot)[None, :] < on[:, None]
    want = np.where(used, oc, 0)[idx]
    assert np.array_equal(cg[good], want[good]) and not cg[~good].any() and s[-1] == nc[-1] == 0
