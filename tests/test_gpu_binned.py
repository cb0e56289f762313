"""The binned kernels on the reference's own calls.  A batch of up to 98,304 tasks
runs a wave per task under every band policy (up to 20,480 for CIGARs), so the
fixtures as they stand reach no pair, lane, group or frame kernel.  Here they do:
as timed calls, which are binned whatever their size, and repeated past those
sizes."""
import numpy as np
import pytest

import cfg0_cases as K
from conftest import EXT_GOLDEN, GLB_GOLDEN, golden_ext, golden_glb
from oracle import oracle as O
from test_gpu_extend import scoring_of
from test_gpu_gpair import repeat as repeat_glb
from test_gpu_pair import repeat

pytestmark = pytest.mark.gpu
DIRECT_MAX, GLB_DIRECT_MAX, GLB_PAIR_MIN = 98304, 20480, 131072
FORMS = ["plain", "learned", "f24", "f40", "f80", "f144"]


@pytest.fixture
def fresh():
    from bsbolt_amd.bsx import Engine
    e = Engine(0)
    yield e
    e.close()


def set_form(e, form):
    from bsbolt_amd import band, bsx
    if form == "learned":
        e.set_band_model(band.load_model())
        e.set_band_policy(bsx.BAND_LEARNED)
    elif form != "plain":
        e.set_band_policy(bsx.BAND_FIXED, FORMS.index(form) - 2)


def check(got, want, idx, what):
    for k in K.FIELDS:
        bad = np.nonzero(got[k] != want[k][idx])[0]
        assert len(bad) == 0, f"{what}: {k} differs at {len(bad)} tasks, first {bad[:8]}"


def run_binned(e, t, sc, want, form, what):
    """As a timed call of its own size, and repeated past the unbinned sizes."""
    e.set_kernel_timing(1)
    check(e.extend(t, sc), want, slice(None), f"{what}, timed")
    ms, calls = e.kernel_times()
    e.set_kernel_timing(0)
    assert calls == 1 and (ms[:11] > 0).any()
    if form not in ("plain", "learned"):
        assert ms[11 + FORMS.index(form) - 2] > 0
    b, idx = repeat(t, DIRECT_MAX + 1 + len(t))
    check(e.extend(b, sc), want, idx, f"{what}, {len(b)} tasks")


@pytest.mark.parametrize("form", FORMS)
def test_binned_kernels_equal_every_reference_call(fresh, form):
    t, sc, ref = K.ext_tasks()
    set_form(fresh, form)
    run_binned(fresh, t, scoring_of(sc), ref, form, form)


@pytest.mark.parametrize("form", ["plain", "f24", "f40", "f80", "f144"])
@pytest.mark.parametrize("name", EXT_GOLDEN)
def test_binned_kernels_on_reference_golden(fresh, name, form):
    t, sc, ref = golden_ext(name)
    set_form(fresh, form)
    run_binned(fresh, t, scoring_of(sc), ref, form, f"{name}, {form}")


@pytest.mark.parametrize("form", ["f40", "f80", "f144"])
def test_frame_kernels_random_scorings(fresh, form):
    """Other gap costs (general e, asymmetric o/e) and N bases, as test_gpu_band has them."""
    from bsbolt_amd.bsx import Scoring
    from bsbolt_amd.tasks import random_ext_tasks
    b = random_ext_tasks(6000, seed=39 + FORMS.index(form), qmax=256, h0max=80, w_choices=(16, 40, 100, 200),
                         eb_choices=(0, 5, 30), n_frac=0.01)
    set_form(fresh, form)
    for sc in (dict(o_del=6, e_del=1, o_ins=6, e_ins=1, zdrop=100), dict(o_del=5, e_del=2, o_ins=3, e_ins=1, zdrop=50),
               dict(o_del=4, e_del=3, o_ins=7, e_ins=2, zdrop=0)):
        want, _ = O.extend2_batch(b, nthreads=16, scoring=sc)
        run_binned(fresh, b, Scoring.make(**sc), want, form, f"{form}, {sc}")


@pytest.mark.parametrize("table", [[16, 16, 1, 0], [64, 32, 0, 1], [128, 64, 1, 1]], ids=str)
@pytest.mark.parametrize("form", FORMS)
def test_binned_kernels_with_every_table(fresh, form, table):
    from bsbolt_amd.bsx import Scoring
    from bsbolt_amd.tasks import random_ext_tasks
    t = random_ext_tasks(20000, seed=91, qmax=200, h0max=120, w_choices=(16, 100), n_frac=0.001)
    want, _ = O.extend2_batch(t, nthreads=16)
    fresh.set_tuning(table)
    set_form(fresh, form)
    run_binned(fresh, t, Scoring.make(), want, form, f"{form}, {table}")


@pytest.mark.parametrize("name", GLB_GOLDEN)
def test_binned_cigar_kernels_on_reference_golden(engine, name):
    t, sc, score, ncig, cig = golden_glb(name)
    slot = cig.shape[1]
    used = np.arange(slot)[None, :] < np.maximum(ncig, 0)[:, None]
    want = np.where(used, cig, 0)
    from bsbolt_amd.bsx import Scoring
    s_ = Scoring.make(mat=sc["mat"], o_del=sc["o_del"], e_del=sc["e_del"], o_ins=sc["o_ins"], e_ins=sc["e_ins"])
    for n in (GLB_DIRECT_MAX + 1 + len(t), GLB_PAIR_MIN + len(t)):
        b, idx = repeat_glb(t, n)
        s, nc, cg = engine.global_(b, s_, slot=slot)
        assert np.array_equal(s, score[idx]) and np.array_equal(nc, ncig[idx]), n
        assert np.array_equal(np.where(used[idx], cg, 0), want[idx]), n
