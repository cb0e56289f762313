"""Performance cases of libbsx: the calls a bisulfite aligner makes on the GPU.

A case is a dict of plain values.  `call` names the entry point it goes
through:

  scalar   bsx.ksw_extend2, one call (the scalar drop-in's Python form)
  host     Engine.extend, numpy arrays in and out (a chunk of an aligner's round)
  device   Engine.extend_device, the batch resident in device memory
  graph    a captured Engine.extend_device batch, replayed (streamed chunks)
  glb_host Engine.global_, numpy arrays in and out (one CIGAR try round)
  glb_dev  Engine.global_device (the CIGAR pass of a resident batch)
  md       Engine.md_device (NM, MD:Z, XB:Z of final CIGARs)

`reads` names the read set the tasks come from (sizes as the named workloads
of bsbolt_amd.workload, scaled), `n` is the number of tasks of one pass, and
`policy` the band policy of the extension (plain kernels, the 24-column frame
for every task, or the trained predictor).

Extension batches hold the ksw_extend2 calls mem_chain2aln makes for simulated
bisulfite reads: the producer's rounds run on the GPU, and its batch is
repeated (each copy with sequence memory of its own) or thinned to n tasks.

torch is imported before libbsx.so is loaded: both then use the one HIP
runtime torch brings, so torch tensors can be handed to libbsx by address.
"""
import math

import numpy as np
import torch

from bsbolt_amd import bsx
from bsbolt_amd import workload as W
from bsbolt_amd.tasks import EXT_FIELDS, GLB_FIELDS, RESULT_FIELDS, ExtTasks, GlbTasks

# Read sets: workload, extension tasks per fragment, and the mean sequence
# bytes and DP cells of one of its ksw_extend2 calls (used by work()).
READS = {
    "se100": dict(cfg=W.CONFIGS["cfg0"], per_frag=1.77, seq=106, cells=630),
    "pe150": dict(cfg=W.CONFIGS["cfg1"], per_frag=3.89, seq=172, cells=1389),
    "se250": dict(cfg=W.CONFIGS["cfg3"], per_frag=2.81, seq=325, cells=6150),
    "rrbs": dict(cfg=W.CONFIGS["cfg4"], per_frag=1.65, seq=65, cells=367),
    # long reads with the 250 bp set's error rates: flanks up to the longest query the library takes
    "se2000": dict(cfg=W.SimConfig(1_000_000, 5, 1_000_000, 105, read_len=2000, sub=0.01, indel=0.005,
                                   geometric_indels=True),
                   per_frag=3.32, seq=2060, cells=101_000),
}
POOL = 78_000         # distinct tasks of a large batch; it is repeated beyond that
POOL_LONG = 2_500     # the same for 2 kb reads
CIGAR_POOL = 40_000   # distinct ksw_global2 tasks
MD_POOL = 50_000      # distinct regions of the NM/MD/XB pass
MD_GENOME = 1_000_000
MD_FLAT = 180         # bytes of a 150-base region's CIGAR, strings and counters


def listed():
    return [
        # one flank through the scalar drop-in: a call site that was not batched
        dict(name="scalar_call", call="scalar", reads="pe150", n=1, policy="plain"),
        # a few hundred resident tasks: one small chunk of reads, the latency of a call
        dict(name="ext_small", call="device", reads="pe150", n=500, policy="plain"),
        # a round of 100 bp single-end reads handed over in host memory
        dict(name="ext_host_se100", call="host", reads="se100", n=20_003, policy="plain"),
        # the whole 1M-pair 2x150 bp run resident in HBM: the benchmark's batch, plain kernels
        dict(name="ext_pe150", call="device", reads="pe150", n=3_900_927, policy="plain"),
        # the same reads, a quarter of them, in the form the benchmark quotes (24-column frame)
        dict(name="ext_pe150_frame", call="device", reads="pe150", n=975_231, policy="frame"),
        # the trained band predictor on an odd-sized batch of them
        dict(name="ext_pe150_learned", call="device", reads="pe150", n=500_009, policy="learned"),
        # 250 bp reads with indels: long flanks, wide bands
        dict(name="ext_se250", call="device", reads="se250", n=351_491, policy="plain"),
        # RRBS reads of 40-100 bp streamed as captured chunks of 262,144 tasks
        dict(name="ext_rrbs_graph", call="graph", reads="rrbs", n=262_144, policy="plain"),
        # 2 kb reads: the longest queries the library takes
        dict(name="ext_se2000", call="device", reads="se2000", n=4_001, policy="plain"),
        # the CIGAR pass of the 150 bp run, resident
        dict(name="cigar_pe150", call="glb_dev", reads="pe150", n=596_416, policy="plain"),
        # one CIGAR try round of a read chunk, host memory
        dict(name="cigar_host_pe150", call="glb_host", reads="pe150", n=9_319, policy="plain"),
        # NM / MD:Z / XB:Z of 150 bp regions
        dict(name="md_pe150", call="md", reads="pe150", n=400_009, policy="plain"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["scalar", "host", "device", "device", "device", "graph", "glb_dev", "glb_host", "md"])
    policy, reads = "plain", rng.choice(["se100", "pe150", "se250", "rrbs"])
    if call == "scalar":
        return dict(call=call, reads=reads, n=1, policy=policy, pick=rng.randrange(1000))
    if call == "host":
        n = _log_uniform(rng, 200, 200_000)
    elif call == "graph":
        n = _log_uniform(rng, 4_000, 262_144)
    elif call == "device":
        policy = rng.choice(["plain", "plain", "frame", "learned"])
        if policy == "plain" and rng.random() < 0.2:
            reads = "se2000"
        cap = 3_900_927 * READS["pe150"]["cells"] / READS[reads]["cells"]
        n = _log_uniform(rng, 300, min(3_900_927, cap, 8_000 if reads == "se2000" else cap))
    elif call == "glb_dev":
        reads = rng.choice(["se100", "pe150", "se250"])
        n = _log_uniform(rng, 300, 300_000 if reads == "se250" else 596_416)
    elif call == "glb_host":
        reads = rng.choice(["se100", "pe150", "se250"])
        n = _log_uniform(rng, 100, 40_000)
    else:
        reads = rng.choice(["se100", "pe150", "se250"])
        n = _log_uniform(rng, 500, 800_000)
    return dict(call=call, reads=reads, n=n, policy=policy)


# ---- engines: a program keeps one per band policy ----

_engines = {}


def _engine(policy):
    if policy not in _engines:
        e = bsx.Engine(0)
        if policy == "frame":
            e.set_band_policy(bsx.BAND_FIXED, 0)
        elif policy == "learned":
            from bsbolt_amd import band
            e.set_band_model(band.load_model())
            e.set_band_policy(bsx.BAND_LEARNED)
        _engines[policy] = e
    return _engines[policy]


# ---- inputs ----

def _ext_pool(reads, want, seed):
    """About `want` distinct ksw_extend2 calls of the read set (host arrays)."""
    import dataclasses
    r = READS[reads]
    base = r["cfg"]
    frags = max(64, int(math.ceil(1.1 * want / r["per_frag"])))
    cfg = base.scaled(min(1.0, frags / base.n_frag))
    cfg = dataclasses.replace(cfg, n_frag=frags, read_seed=1000 + int(seed), genome_seed=int(seed) % 1009,
                              genome_len=min(cfg.genome_len, 2_000_000))
    wl = W.Workload(cfg)
    try:
        eng = _engine("plain")
        batch, _, _, _ = wl.build_ext_batch(lambda t: eng.extend(t, cells=False))
    finally:
        wl.close()
    return batch


def _thin(p, n):
    return (np.arange(n, dtype=np.int64) * p) // n


def _repeat(arrays, n, fields):
    """The batch on the GPU, thinned or repeated to n tasks; every copy has its
    own sequence bytes.  Returns a dict of tensors."""
    p = len(arrays["qlen"])
    dev = {}
    if n <= p:
        idx = _thin(p, n)
        for k in fields:
            a = arrays[k] if k in ("query", "target") else arrays[k][idx]
            dev[k] = torch.from_numpy(np.ascontiguousarray(a).view(np.int64 if k.endswith("_off") else a.dtype)).cuda()
        return dev
    reps = -(-n // p)
    for k in fields:
        a = arrays[k]
        t = torch.from_numpy(np.ascontiguousarray(a).view(np.int64 if k.endswith("_off") else a.dtype)).cuda()
        if k in ("query", "target"):
            dev[k] = t.repeat(reps)
        elif k.endswith("_off"):
            step = len(arrays["query" if k == "q_off" else "target"])
            dev[k] = (torch.arange(reps, device="cuda")[:, None] * step + t[None, :]).reshape(-1)[:n].contiguous()
        else:
            dev[k] = t.repeat(reps)[:n].contiguous()
    return dev


def _host_thin(batch, n, cls, fields):
    """n of the batch's tasks as a host batch of its own (repeated if it has fewer)."""
    p = len(batch)
    idx = _thin(p, n) if n <= p else np.arange(n, dtype=np.int64) % p
    a = {k: getattr(batch, k) for k in fields}
    return cls(*[a[k] if k in ("query", "target") else a[k][idx] for k in fields])


def _glb_pool(reads, m, seed):
    """ksw_global2 calls of mem_reg2aln for reads whose region needs a DP (a few
    substitutions or an indel): the band follows from the region's score."""
    rng = np.random.default_rng([7, int(seed)])
    rl = READS[reads]["cfg"].read_len
    long_indel = READS[reads]["cfg"].geometric_indels
    k = 2 * m + 64
    ql = np.where(rng.random(k) < 0.8, rl, rng.integers(30, rl + 1, k)).astype(np.int64)
    ins = np.minimum(rng.geometric(0.25, k), 30) if long_indel else rng.integers(1, 4, k)
    kind = rng.choice(3, k, p=[0.4, 0.3, 0.3])          # no indel, insertion, deletion
    gap = np.where(kind == 0, 0, np.minimum(ins, ql // 4))
    nsub = np.where(kind == 0, 3 + rng.poisson(0.7, k), rng.poisson(0.005 * ql))
    tl = ql + np.where(kind == 2, gap, 0) - np.where(kind == 1, gap, 0)
    score = np.maximum(ql - np.where(kind == 1, gap, 0) - 5 * nsub - np.where(gap > 0, 6 + gap, 0), 1)
    w2 = np.maximum(W.infer_bw(ql, tl, score, 1, 6, 1), 0)
    w2 = np.minimum(w2 * np.where(rng.random(k) < 0.04, 2, 1), 400)  # a second try doubles it
    keep = np.flatnonzero((w2 > 0) | (ql != tl))[:m]
    ql, tl, gap, kind, nsub, w2 = (x[keep] for x in (ql, tl, gap, kind, nsub, w2))
    w = W.cigar_band(w2, ql, tl)
    n = len(ql)
    toff = np.zeros(n, np.int64)
    toff[1:] = np.cumsum(tl)[:-1]
    qoff = np.zeros(n, np.int64)
    qoff[1:] = np.cumsum(ql)[:-1]
    letters = np.array([0, 2, 3, 3], np.uint8)  # converted reference: A, G, T (C reads as T)
    target = letters[rng.choice(4, int(tl.sum()), p=[0.295, 0.205, 0.205, 0.295])]
    own = np.repeat(np.arange(n), ql)
    x = np.arange(int(ql.sum())) - np.repeat(qoff, ql)
    at = (ql * (0.1 + 0.8 * rng.random(n))).astype(np.int64)[own]  # where the indel sits
    src = x + np.where((kind[own] == 2) & (x >= at), gap[own], 0) - np.where((kind[own] == 1) & (x >= at), gap[own], 0)
    fresh = (kind[own] == 1) & (x >= at) & (x < at + gap[own])
    query = target[toff[own] + np.clip(src, 0, tl[own] - 1)]
    noise = rng.integers(0, 4, len(query)).astype(np.uint8)
    sub = rng.random(len(query)) < (nsub / np.maximum(ql, 1))[own]
    query = np.where(fresh | sub, noise, query).astype(np.uint8)
    return GlbTasks(query, qoff, ql, target, toff, tl, w)


def _md_pool(reads, m, seed):
    """Regions with their final CIGARs and reads as sequenced, on both strands
    of both reference copies: mostly one M, a sixth with an indel."""
    rng = np.random.default_rng([11, int(seed)])
    rl = READS[reads]["cfg"].read_len
    G = MD_GENOME
    genome = W.make_genome(G, int(seed) % 1013)
    l_pac = 2 * G
    both = np.concatenate([genome, genome])
    ql = np.where(rng.random(m) < 0.85, rl, rng.integers(30, rl + 1, m)).astype(np.int64)
    kind = rng.choice(3, m, p=[0.84, 0.08, 0.08])
    gap = np.where(kind == 0, 0, rng.integers(1, 4, m))
    rlen = ql + np.where(kind == 2, gap, 0) - np.where(kind == 1, gap, 0)
    at = 10 + ((ql - 20 - gap) * rng.random(m)).astype(np.int64)
    copy = rng.integers(0, 4, m)  # which of the four copies the region lies on
    rb = copy * G + 8 + (rng.random(m) * (G - 2 * rl - 64)).astype(np.int64)
    re = rb + rlen
    fwd = rb < l_pac
    crick = ((rb >= G) & (rb < l_pac)) | (rb >= G + l_pac)
    own = np.repeat(np.arange(m), ql)
    off = np.zeros(m, np.int64)
    off[1:] = np.cumsum(ql)[:-1]
    x = np.arange(int(ql.sum())) - off[own]          # index in walking order
    y = x + np.where((kind[own] == 2) & (x >= at[own]), gap[own], 0) \
        - np.where((kind[own] == 1) & (x >= at[own] + gap[own]), gap[own], 0)
    y = np.clip(y, 0, rlen[own] - 1)
    pos = np.where(fwd[own], rb[own] + y, re[own] - 1 - y)  # the reverse strand is walked backwards
    c = np.where(pos < l_pac, both[np.where(pos < l_pac, pos, 0)],
                 3 - both[np.where(pos < l_pac, 0, 2 * l_pac - 1 - pos)]).astype(np.uint8)
    ref_base, methyl = np.where(crick[own], 2, 1), np.where(crick[own], 0, 3)
    c = np.where((c == ref_base) & (rng.random(len(c)) < 0.85), methyl, c)
    c = np.where(rng.random(len(c)) < 0.006, rng.integers(0, 4, len(c)), c)
    fresh = (kind[own] == 1) & (x >= at[own]) & (x < at[own] + gap[own])
    c = np.where(fresh, rng.integers(0, 4, len(c)), c).astype(np.uint8)
    oquery = np.empty_like(c)
    oquery[off[own] + np.where(fwd[own], x, ql[own] - 1 - x)] = c
    cig = np.zeros((m, 3), np.uint32)
    one = kind == 0
    cig[:, 0] = np.where(one, ql, at) << 4
    cig[:, 1] = np.where(one, 0, gap << 4 | np.where(kind == 1, 1, 2))
    cig[:, 2] = np.where(one, 0, (ql - at - np.where(kind == 1, gap, 0)) << 4)
    return dict(opac=W.pack2(both), l_pac=l_pac, crick_l=G, rb=rb, re=re, oquery=oquery, oq_off=off,
                l_query=ql.astype(np.int32), n_cigar=np.where(one, 1, 3).astype(np.int32), cigar=cig)


def prepare(case, seed):
    n, reads, call = case["n"], case["reads"], case["call"]
    st = {"call": call, "eng": _engine(case["policy"]), "n": n}
    if call == "scalar":
        b = _ext_pool(reads, 500, seed)
        order = np.argsort(b.qlen, kind="stable")
        i = int(order[(case.get("pick", 700) * len(b)) // 1000])
        st["args"] = (int(b.qlen[i]), b.query_of(i), int(b.tlen[i]), b.target_of(i), 5, bsx.fill_scmat(), 6, 1, 6, 1,
                      int(b.w[i]), int(b.end_bonus[i]), 100, int(b.h0[i]))
    elif call in ("host", "device", "graph"):
        pool = _ext_pool(reads, min(n, POOL_LONG if reads == "se2000" else POOL), seed)
        if call == "host":
            st["tasks"] = _host_thin(pool, n, ExtTasks, EXT_FIELDS)
            return st
        dev = _repeat(pool.arrays(), n, EXT_FIELDS)
        out = {k: torch.zeros(n, dtype=torch.int32, device="cuda") for k in RESULT_FIELDS}
        out["cells"] = torch.zeros(n, dtype=torch.int64, device="cuda")
        st["keep"], st["out"] = dev, out
        st["ptrs"] = {k: v.data_ptr() for k, v in {**dev, **out}.items()}
        st["ptrs"]["n"] = n
        torch.cuda.synchronize()
        if call == "graph":
            st["graph"] = st["eng"].capture_extend(st["ptrs"])
    elif call in ("glb_host", "glb_dev"):
        pool = _glb_pool(reads, min(n, CIGAR_POOL), seed)
        if call == "glb_host":
            st["tasks"] = _host_thin(pool, n, GlbTasks, GLB_FIELDS)
            return st
        dev = _repeat({k: getattr(pool, k) for k in GLB_FIELDS}, n, GLB_FIELDS)
        slot = int((pool.qlen + pool.tlen).max())
        out = {"score": torch.zeros(n, dtype=torch.int32, device="cuda"),
               "n_cigar": torch.zeros(n, dtype=torch.int32, device="cuda"),
               "cigar": torch.zeros((n, slot), dtype=torch.int32, device="cuda")}
        st["keep"], st["out"] = dev, out
        st["ptrs"] = {k: v.data_ptr() for k, v in {**dev, **out}.items()}
        st["ptrs"].update(n=n, cigar_slot=slot)
        torch.cuda.synchronize()
    else:
        p = _md_pool(reads, min(n, MD_POOL), seed)
        m = len(p["rb"])
        reps = -(-n // m)
        idx = _thin(m, n) if n <= m else None
        dev = {"opac": torch.from_numpy(p["opac"]).cuda()}
        oq = torch.from_numpy(p["oquery"]).cuda()
        dev["oquery"] = oq if idx is not None else oq.repeat(reps)
        for k in ("rb", "re", "oq_off", "l_query", "n_cigar", "cigar"):
            if idx is not None:
                a = np.ascontiguousarray(p[k][idx])
                dev[k] = torch.from_numpy(a.view(np.int32) if k == "cigar" else a).cuda()
                continue
            t = torch.from_numpy(p[k].view(np.int32) if k == "cigar" else p[k]).cuda()
            if k == "oq_off":
                dev[k] = (torch.arange(reps, device="cuda")[:, None] * len(p["oquery"]) + t[None, :]).reshape(-1)[:n]
            else:
                dev[k] = t.repeat(*([reps] + [1] * (t.dim() - 1)))[:n]
            dev[k] = dev[k].contiguous()
        ls = int(p["l_query"].max())
        md_slot, xb_slot = 4 * ls + 4 * 3 + 16, 4 * ls + 16
        out = {"md": torch.zeros((n, md_slot), dtype=torch.uint8, device="cuda"),
               "xb": torch.zeros((n, xb_slot), dtype=torch.uint8, device="cuda"),
               "meth": torch.zeros((n, 4), dtype=torch.int32, device="cuda")}
        for k in ("md_len", "xb_len", "nm", "status"):
            out[k] = torch.zeros(n, dtype=torch.int32, device="cuda")
        st["keep"], st["out"] = dev, out
        st["ptrs"] = {k: v.data_ptr() for k, v in {**dev, **out}.items()}
        st["ptrs"].update(n=n, l_pac=p["l_pac"], crick_l=p["crick_l"], cigar_slot=3, md_slot=md_slot, xb_slot=xb_slot)
        torch.cuda.synchronize()
    return st


# ---- one pass ----

def run(state):
    call, eng = state["call"], state["eng"]
    if call == "scalar":
        return bsx.ksw_extend2(*state["args"])
    if call == "host":
        return eng.extend(state["tasks"])
    if call == "device":
        eng.extend_device(state["ptrs"])
        return state["out"]
    if call == "graph":
        state["graph"].launch()
        return state["out"]
    if call == "glb_host":
        return eng.global_(state["tasks"])
    if call == "glb_dev":
        eng.global_device(state["ptrs"])
        return state["out"]
    eng.md_device(state["ptrs"])
    return state["out"]


# ---- what a pass cannot do without ----

def work(case):
    """Bytes: sequences, the per-task arrays and the results once.  Operations:
    12 integer operations per cell of the reference's band (ksw.c:433-447 for
    the extension, ksw.c:548-565 for the global kernel), one per base of the
    string layer."""
    n, r = case["n"], READS[case["reads"]]
    if case["call"] in ("scalar", "host", "device", "graph"):
        return {"bytes": n * (r["seq"] + 36 + 32), "flops": 12 * n * r["cells"]}
    rl = r["cfg"].read_len
    if case["call"] in ("glb_host", "glb_dev"):
        return {"bytes": n * (2 * 0.93 * rl + 28 + 8 + 3 * 4), "flops": 12 * n * 0.93 * rl * 19}
    return {"bytes": n * (1.25 * rl + MD_FLAT), "flops": n * rl}
