"""Autotuner of the extension kernels' launch table.

Sweeps, on the GPU, the knobs of the tuning table (include/bsx.h,
bsx_set_tuning): the chunk of the plain group kernels, descriptors per block of the
frame group kernels, and the group shape of the two query-length bins that have
alternatives (65-96 and 97-128 bases: 16 lanes x 6/8 columns or 32 lanes x 3/4
columns).  Coordinate descent from the current table: each knob in turn takes
the value with the lowest step time, if that is 2% below the present value's, and
every candidate's outputs are checked equal to the default table's.  The plain
knobs act on tasks outside the packed kernels' range, so they are swept in the
plain form on the workload's tasks with higher start scores, as the flanks of long
reads have; the frame knob in the 24-column frame form with plain fallback, on the
workload as it is and on a quarter of it.  The winner is cached in bsbolt_amd/tune.json under the
device's key ("<gfx arch>/<CU count>"), which bsx_create loads.

    python -m bsbolt_amd.tune [--workload cfg1] [--scale 0.5] [--steps 5]
"""
import argparse
import dataclasses
import json
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
CACHE = os.path.join(HERE, "tune.json")
KNOBS = (("tpb_plain", 0, (16, 32, 64, 128)), ("shape_var_65_96", 2, (0, 1)),
         ("shape_var_97_128", 3, (0, 1)), ("tpb_narrow", 1, (16, 32, 64)))


def _time(eng, ptrs, steps, reps=3):
    best = float("inf")
    for _ in range(reps):
        eng.extend_device(ptrs)
        eng.sync()
        eng.timer_start()
        for _ in range(steps):
            eng.extend_device(ptrs)
        best = min(best, eng.timer_stop() / steps)
    return best


def outside_range(batch):
    """The batch with start scores that the packed kernels do not hold."""
    return dataclasses.replace(batch, h0=batch.h0 + 600)


def tune(eng, batch, steps=5, log=print):
    """Returns (table, record) for the resident batch."""
    from . import bsx
    from .tasks import RESULT_FIELDS
    n = len(batch)
    outs = {k: eng.empty((n,), np.int32) for k in RESULT_FIELDS}
    table = list(eng.get_tuning()[0])  # the cached one, where there is one

    def resident(b):
        keep, ptrs = eng.tasks_to_device(b)
        ptrs.update({k: v.ptr for k, v in outs.items()})
        ptrs["n"] = n
        eng.set_tuning(None)
        eng.extend_device(ptrs)
        eng.sync()
        return keep, ptrs, {k: v.numpy() for k, v in outs.items()}

    sets = {"plain": resident(outside_range(batch)), "frame24": resident(batch)}
    eng.set_tuning(None)
    default = eng.get_tuning()[0]
    record = {"sweep": []}

    def form(name):
        eng.set_band_policy(*((bsx.BAND_FIXED, 0) if name == "frame24" else (bsx.BAND_PLAIN, 0)))

    try:
        for name, idx, values in KNOBS:
            which = "frame24" if name == "tpb_narrow" else "plain"
            _, ptrs, ref = sets[which]
            form(which)
            times = {}
            for v in values:
                t = list(table)
                t[idx] = v
                eng.set_tuning(t)
                ms = _time(eng, ptrs, steps)
                if which == "frame24":  # of two sizes, as blocks of many tasks suit the larger alone
                    ms = (ms + 4 * _time(eng, dict(ptrs, n=n // 4), 2 * steps)) / 2
                for k in RESULT_FIELDS:
                    if not np.array_equal(outs[k].numpy(), ref[k]):
                        raise RuntimeError(f"tuning {name}={v} changed output {k}")
                times[v] = ms
                log(f"  {name}={v}: {ms:.3f} ms/step")
            best = min(times, key=times.get)
            if times[best] < 0.98 * times.get(table[idx], float("inf")):
                table[idx] = best
            record["sweep"].append({"knob": name, "ms": {str(k): v for k, v in times.items()},
                                    "chosen": table[idx]})
        for key, tb in (("default_ms", default), ("tuned_ms", table)):
            eng.set_tuning(tb)
            record[key] = {}
            for which, (_, ptrs, _) in sets.items():
                form(which)
                record[key][which] = _time(eng, ptrs, steps)
    finally:
        eng.set_band_policy(bsx.BAND_PLAIN)
    del sets, outs
    return table, record


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--workload", default="cfg1")
    ap.add_argument("--scale", type=float, default=0.5)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--out", default=CACHE)
    args = ap.parse_args()
    from . import bsx
    from .workload import CONFIGS, Workload
    eng = bsx.Engine(0)
    wl = Workload(CONFIGS[args.workload].scaled(args.scale))
    batch = wl.build_ext_batch(lambda t: eng.extend(t, cells=False))[0]
    wl.close()
    key = eng.get_tuning()[2]
    print(f"tuning {key} on {args.workload} x {args.scale}: {len(batch)} tasks", flush=True)
    table, rec = tune(eng, batch, args.steps, log=lambda m: print(m, flush=True))
    cache = json.load(open(args.out)) if os.path.exists(args.out) else {}
    cache[key] = {"bsx_table": table,
                  "workload": f"{args.workload} x {args.scale} ({len(batch)} tasks; plain knobs: start scores + 600)",
                  **rec}
    with open(args.out, "w") as f:
        json.dump(cache, f, indent=1, sort_keys=True)
    print(f"{key}: {table} (default {rec['default_ms']['plain']:.3f} ms, tuned {rec['tuned_ms']['plain']:.3f} ms) "
          f"-> {args.out}", flush=True)
    eng.close()


if __name__ == "__main__":
    sys.exit(main())
