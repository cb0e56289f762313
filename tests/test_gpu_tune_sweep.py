"""The autotuner's sweep of the plain group kernels' knobs runs a batch that is
theirs: under the default scoring the packed kernels take nearly every task."""
import pytest

from test_gpu_pair import repeat

pytestmark = pytest.mark.gpu


def test_the_sweep_reaches_the_tuned_kernels(wl_small):
    from bsbolt_amd import bsx, tune
    from bsbolt_amd.tasks import EXT_FIELDS
    from bsbolt_amd.workload import concat_ext
    e = bsx.Engine(0)
    try:
        e.set_side_streams(False)  # each kernel by itself
        b, _ = repeat(concat_ext(list(wl_small)), 120_000)
        share = {}
        for name, t in (("workload", b), ("sweep", tune.outside_range(b))):
            for _ in range(2):
                e.set_kernel_timing(1)
                e.extend(t)
                ms = e.kernel_times()[0]
            share[name] = float(ms[9:11].sum() / ms[:11].sum())
        assert share["workload"] < 0.2 and share["sweep"] > 0.7, share
        e.set_kernel_timing(0)
        table, rec = tune.tune(e, b, steps=2, log=lambda m: None)
        assert [k["knob"] for k in rec["sweep"]] == [k[0] for k in tune.KNOBS]
        assert all(rec["tuned_ms"][k] < 1.1 * rec["default_ms"][k] for k in ("plain", "frame24")), rec
    finally:
        e.close()
