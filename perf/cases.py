"""The work a user has this framework do, as cases that can be timed.

Four kinds, by use:

  overlap  the daligner command's work: one block against itself (k-mer index,
           both strands' match filter and alignment, the .las file), from
           reads resident in HBM; the .las bytes are the output
  pair     the same for two different blocks (both .las files)
  align    a batch of Local_Alignment tasks held in HBM (mi_la_batch_device)
  trace    Compute_Trace_PTS over a batch of paths (host arrays)
  dust     the DBdust scan of a block (host arrays)
  lasort   LAsort of a .las body (host arrays)

Outputs whose length depends on the data are padded with zeros to a length
that depends on the case alone.  Reads are simulated from the case's seed (marvel_amd.sim's error model: every
read has the case's error, split 9:4:2 into insertions, deletions and
substitutions).  Every output is an integer or a byte of a file format that
is pinned bit for bit, so every tolerance is "exact" and there is no 64-bit
reference to compare with (`exact` gives None).
"""

import ctypes as C
import math
import os
import shutil
import tempfile
import weakref

import numpy as np
import torch

from marvel_amd import dbio, sim
from marvel_amd.align import gen_tasks_device, la_batch_device
from marvel_amd.daligner import HITS_DB, Daligner
from marvel_amd.lib import MiTraceResult, MiTraceTask, lib


def listed():
    overlap = dict(kind="overlap", families=0, mean=10000, sd=6000, err=0.15, kmer=14, hitmin=35, corr=0.70, tspace=100)
    return [
        # a few hundred reads: launches, host synchronisations and small copies decide
        dict(overlap, name="overlap-tiny", genome=40_000, coverage=12.0, mean=3000, sd=1500),
        # the small test genome (200 kbp at 20x), 16-bit traces as -s above 125 gives them
        dict(overlap, name="overlap-small", genome=200_000, coverage=20.0, mean=4000, sd=2000, tspace=200),
        # an ordinary bacterial-plasmid-sized block, odd sizes, longer k-mers
        dict(overlap, name="overlap-1mbp", genome=1_000_003, coverage=30.0, kmer=16),
        # the headline workload: 5 Mbp at 30x, one block of about 158 Mbp
        dict(overlap, name="overlap-5mbp", genome=5_000_000, coverage=30.0),
        # a repeat-rich block: families of 40 copies and tandem repeats, 12 % error
        dict(overlap, name="overlap-repeats", genome=12_000_000, coverage=4.0, families=48, err=0.12),
        # two blocks of a long-read set against each other, 8 % error, -e.75 (both files)
        dict(overlap, name="pair-long-reads", kind="pair", genome=16_000_000, coverage=5.0, families=32, mean=25000,
             sd=20000, err=0.08, corr=0.75),
        # Local_Alignment batches: a handful of calls, an ordinary batch, a large one
        dict(name="align-64", kind="align", tasks=64, lmin=1000, lmax=20000, emin=0.05, emax=0.20, offmax=0, tspace=100),
        dict(name="align-20k", kind="align", tasks=20_000, lmin=1000, lmax=60000, emin=0.10, emax=0.30, offmax=20,
             tspace=100),
        # the batched-aligner workload's model: seeds up to 200 bases off the diagonal
        dict(name="align-400k", kind="align", tasks=400_000, lmin=1000, lmax=60000, emin=0.05, emax=0.20, offmax=200,
             tspace=100),
        # exact alignments between the trace points of some thousand overlaps
        dict(name="trace-4k", kind="trace", tasks=4000, lmin=1000, lmax=20000, emin=0.05, emax=0.25, mode=0),
        # the dust track of a block before it is compared
        dict(name="dust-45mbp", kind="dust", genome=1_500_000, coverage=30.0, window=64, threshold=2.0, mlen=9),
        # the records of a block comparison brought into order
        dict(name="lasort-300k", kind="lasort", records=300_000, reads=15_000, mean=7000),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["overlap", "overlap", "overlap", "overlap", "pair", "align", "align", "align", "trace", "dust",
                       "lasort"])
    if kind in ("overlap", "pair"):
        c = dict(kind=kind, families=0, kmer=rng.choice([14, 14, 14, 15, 16]), hitmin=rng.choice([35, 35, 40, 50]),
                 corr=rng.choice([0.70, 0.70, 0.75]), tspace=rng.choice([100, 100, 100, 80, 126, 200]))
        c["mean"] = int(_log(rng, 3000, 25000))
        c["sd"] = int(c["mean"] * rng.uniform(0.4, 0.8))
        c["err"] = round(rng.uniform(0.06, 0.15), 4)
        if rng.random() < 0.6:   # an iid genome at high coverage
            c["genome"] = max(int(_log(rng, 40_000, 2_500_000)), 4 * c["mean"])
            c["coverage"] = round(rng.uniform(10.0, 30.0), 2)
        else:                    # repeats at the coverage a block of a larger genome has
            c["genome"] = int(_log(rng, 1_000_000, 9_000_000))
            c["coverage"] = round(rng.uniform(3.0, 6.0), 2)
            c["families"] = max(1, c["genome"] // 250_000)
        return c
    if kind == "align":
        emin = round(rng.uniform(0.03, 0.15), 4)
        lmin = int(_log(rng, 500, 4000))
        return dict(kind=kind, tasks=int(_log(rng, 1, 300_000)), lmin=lmin, lmax=int(_log(rng, 2 * lmin, 60000)),
                    emin=emin, emax=round(emin + rng.uniform(0.02, 0.15), 4), offmax=rng.choice([0, 0, 5, 20, 200]),
                    tspace=rng.choice([100, 100, 100, 80, 126, 200]))
    if kind == "trace":
        emin = round(rng.uniform(0.03, 0.12), 4)
        return dict(kind=kind, tasks=int(_log(rng, 1, 4000)), lmin=1000, lmax=int(_log(rng, 2000, 20000)), emin=emin,
                    emax=round(emin + rng.uniform(0.02, 0.13), 4), mode=rng.choice([-1, 0, 1]))
    if kind == "dust":
        return dict(kind=kind, genome=int(_log(rng, 40_000, 1_500_000)), coverage=round(rng.uniform(10.0, 30.0), 2),
                    window=rng.choice([32, 64, 64, 100]), threshold=rng.choice([1.5, 2.0, 2.0, 3.0]),
                    mlen=rng.choice([9, 9, 19]))
    return dict(kind=kind, records=int(_log(rng, 100, 300_000)), reads=int(_log(rng, 100, 30_000)),
                mean=int(_log(rng, 1500, 20000)))


# ---- sizes of padded outputs --------------------------------------------------------


def _mean_len(case):
    lo, hi = case["lmin"], max(case["lmax"], case["lmin"] + 1)
    return (hi - lo) / math.log(hi / lo)   # templates are log-uniform


def _bound(n, mean, worst):
    """A length n values of this mean and worst case never sum beyond."""
    return int(min(n * worst, 1.3 * n * mean + 8 * math.sqrt(n) * worst)) + 64


def _las_bytes(case):
    pairs = case["genome"] * case["coverage"] / case["mean"] * case["coverage"]
    records = 40_000 + 4 * pairs + case["families"] * (64 * case["coverage"]) ** 2
    return int(records * (40 + (2 if case["tspace"] <= 125 else 4) * (case["mean"] / case["tspace"] + 2)))


def _trace_values(case):
    return _bound(case["tasks"], 4 * (1.05 * _mean_len(case) / case["tspace"] + 3),
                  4 * (1.35 * case["lmax"] / case["tspace"] + 3))


# ---- inputs ------------------------------------------------------------------------


def _reads(case, seed):
    length, families = case["genome"], case.get("families", 0)
    if families:
        g = sim.repeat_model_genome(length, seed, families=families)
    else:
        g = sim.random_genome(length, seed)
    err = case.get("err", 0.15)
    return sim.simulate_reads(g, case["coverage"], case.get("mean", 10000), case.get("sd", 6000), 1000, seed + 1000,
                              p_ins=err * 9 / 15, p_del=err * 4 / 15, p_sub=err * 2 / 15, max_len=200_000).reads


def _folder():
    base = "/dev/shm" if os.path.isdir("/dev/shm") and os.access("/dev/shm", os.W_OK) else None
    return tempfile.mkdtemp(prefix="micase_", dir=base)


def _blocks(case, seed, dal, d):
    """The case's reads as a DB in folder d, opened: one block, or two of half the reads each."""
    reads = _reads(case, seed)
    parts = [reads] if case["kind"] != "pair" else [reads[:len(reads) // 2], reads[len(reads) // 2:]]
    blocks = []
    for i, part in enumerate(parts):
        name = "P%d" % (i + 1)
        dbio.write_db(os.path.join(d, name), part, size_mbp=100_000)
        b = dal.open_block(os.path.join(d, name + ".1"))
        if i:   # the second part's reads follow the first's, as in one DB
            b.part, b.ufirst = i + 1, len(parts[0])
        blocks.append(b)
        for f in (name + ".db", "." + name + ".idx", "." + name + ".bps"):
            os.remove(os.path.join(d, f))
    return blocks


def _release(dal, blocks, devs, specs, d):
    for x in devs:
        dal.free_index(x)
    for x in specs:
        dal.h.Free_Align_Spec(x)
    for b in blocks:
        dal.close_block(b)
    shutil.rmtree(d, ignore_errors=True)


class State:
    pass


def _prepare_overlap(case, seed, s):
    s.dal = dal = Daligner()
    dal.configure(nthreads=8, mem_limit_gb=32, minover=2000, symmetric=1)
    dal.set_filter_params(case["kmer"], 6, 0, case["hitmin"])
    s.dir = _folder()
    s.blocks = _blocks(case, seed, dal, s.dir)
    freq = list(s.blocks[0].freq)
    s.spec = dal.new_align_spec(case["corr"], case["tspace"], freq, nthreads=8)
    s.devs = [dal.block_device(b) for b in s.blocks]     # reads packed and resident in HBM
    s.comp = dal.complement_header(s.blocks[-1])
    for b in s.blocks:
        os.makedirs(os.path.join(s.dir, "001_%05d" % b.part), exist_ok=True)
    dal.synchronize()
    s.end = weakref.finalize(s, _release, dal, list(s.blocks), list(s.devs), [s.spec], s.dir)


def _prepare_align(case, seed, s):
    s.tasks = gen_tasks_device(case["tasks"], seed, case["lmin"], case["lmax"], case["emin"], case["emax"],
                               case["offmax"])


def _prepare_trace(case, seed, s):
    dt = gen_tasks_device(case["tasks"], seed, case["lmin"], case["lmax"], case["emin"], case["emax"], 0)
    r = la_batch_device(dt, tspace=100)
    f, arena, t = r.fields(), r.traces(), dt.task_fields()
    keep = np.flatnonzero((f["status"] == 0) & (f["aepos"] > f["abpos"]) & (f["bepos"] > f["bbpos"]))
    f, t = f[keep], t[keep]
    s.packed = dt.words()
    s.n = len(keep)
    tasks = np.zeros(max(s.n, 1), dtype=np.dtype(MiTraceTask))
    ll = np.ascontiguousarray(t[:, :4]).view(np.int64)
    n = f["atlen"].astype(np.int64)
    first = np.cumsum(n) - n
    total = int(n.sum())
    s.points = arena[np.repeat(f["atrace"] - first, n) + np.arange(total)] if total else np.zeros(1, np.uint16)
    if s.n:
        tasks["aword"], tasks["bword"], tasks["alen"], tasks["blen"] = ll[:, 0], ll[:, 1], t[:, 4], t[:, 5]
        for k in ("abpos", "bbpos", "aepos", "bepos"):
            tasks[k] = f[k]
        tasks["tlen"], tasks["points"] = f["atlen"], first
    s.trace_tasks = tasks
    s.results = np.zeros(case["tasks"], dtype=np.dtype(MiTraceResult))
    s.trace = np.zeros(_bound(case["tasks"], 1.1 * case["emax"] * _mean_len(case) + 16,
                              1.35 * case["emax"] * case["lmax"] + 64), dtype=np.int32)


def _prepare_dust(case, seed, s):
    s.dal = dal = Daligner()
    dal.h.mi_dust.argtypes = [C.POINTER(HITS_DB), C.c_int, C.c_double, C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    s.dir = _folder()
    tandems = [(2 + (7 * i + seed) % 30, 200 + 37 * i) for i in range(1 + case["genome"] // 100_000)]
    g = sim.repeat_genome(case["genome"], seed, tandems=tandems)
    reads = sim.simulate_reads(g, case["coverage"], 10000.0, 6000.0, 1000, seed + 1000).reads
    dbio.write_db(os.path.join(s.dir, "P1"), reads, size_mbp=100_000)
    s.blocks = [dal.open_block(os.path.join(s.dir, "P1.1"))]
    bases = case["genome"] * case["coverage"]
    s.anno = np.zeros(64 + int(bases / 8000), dtype=np.int64)
    s.points = np.zeros(max(int(s.blocks[0].totlen), int(bases / 8)) + 64, dtype=np.int32)
    s.npoints = int(bases / 8) + 64
    s.end = weakref.finalize(s, _release, dal, list(s.blocks), [], [], s.dir)


def _prepare_lasort(case, seed, s):
    s.dal = dal = Daligner()
    dal.h.mi_las_sort.argtypes = [C.c_void_p, C.c_longlong, C.c_longlong, C.c_int, C.c_void_p,
                                  C.POINTER(C.c_longlong)]
    rng = np.random.default_rng(seed)
    n = case["records"]
    span = np.maximum(rng.exponential(case["mean"], n), 1000).astype(np.int64)
    rec = np.zeros(n, dtype=dbio.LAS_REC)
    rec["tlen"] = 2 * (span // 100 + 1)
    rec["diffs"] = (span * 0.27).astype(np.int32)
    rec["abpos"] = rng.integers(0, 8000, n)
    rec["bbpos"] = rng.integers(0, 8000, n)
    rec["aepos"], rec["bepos"] = rec["abpos"] + span, rec["bbpos"] + span
    rec["flags"] = rng.integers(0, 2, n)
    rec["aread"], rec["bread"] = rng.integers(0, case["reads"], n), rng.integers(0, case["reads"], n)
    size = 40 + rec["tlen"].astype(np.int64)
    off = np.cumsum(size) - size
    s.body = rng.integers(10, 60, int(size.sum()), dtype=np.uint8)
    head = rec.view(np.uint8).reshape(n, 40)
    for c0 in range(0, n, 65536):
        o = off[c0:c0 + 65536]
        s.body[o[:, None] + np.arange(40)] = head[c0:c0 + 65536]
    s.n = n
    s.out = np.zeros(n * 44 + _bound(n, case["mean"] / 50 + 20, case["mean"] / 4 + 20), dtype=np.uint8)


def prepare(case, seed):
    s = State()
    s.case = dict(case)
    {"overlap": _prepare_overlap, "pair": _prepare_overlap, "align": _prepare_align, "trace": _prepare_trace,
     "dust": _prepare_dust, "lasort": _prepare_lasort}[case["kind"]](case, seed, s)
    return s


# ---- one pass ------------------------------------------------------------------------


def _las(path, size):
    """A .las file's bytes (mapped, the name given back), the file lengthened to `size`."""
    if os.path.getsize(path) > size:
        raise RuntimeError("%s: more than %d bytes" % (path, size))
    os.truncate(path, size)
    m = np.memmap(path, dtype=np.uint8, mode="r")
    os.remove(path)
    return m


def _run_overlap(s):
    cwd = os.getcwd()
    os.chdir(s.dir)
    try:
        s.dal.compare_self(s.blocks[0], s.spec, 1, "P.1", dev=s.devs[0], cA=s.comp)
        return _las("001_00001/P.1.P.1.las", _las_bytes(s.case))
    finally:
        os.chdir(cwd)


def _run_pair(s):
    """Block A against another block B, as `daligner A B` does (dalign/daligner.c:994-1024)."""
    dal, (A, B) = s.dal, s.blocks
    na, nb = C.create_string_buffer(b"P.1"), C.create_string_buffer(b"P.2")
    cwd = os.getcwd()
    os.chdir(s.dir)
    try:
        a, b = dal.sort_kmers_device(s.devs[0]), dal.sort_kmers_device(s.devs[1])
        c = dal.sort_kmers_complement(b, s.comp)
        dal.match_filter(na, A, nb, B, a, b, 0, s.spec)         # consumes b
        dal.match_filter(na, A, nb, s.comp, a, c, 1, s.spec)    # consumes c
        dal.free_index(a)
        dal.write_overlap_buffer(s.spec, 1, na, nb, A.ufirst + A.nreads - 1)
        dal.reset_overlap_buffer(s.spec)
        return [_las("001_00001/P.1.P.2.las", _las_bytes(s.case)), _las("001_00002/P.2.P.1.las", _las_bytes(s.case))]
    finally:
        os.chdir(cwd)


class _View:
    """A device buffer of the library as an array torch can take without a copy."""

    def __init__(self, buf, count, typestr):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (buf.ptr, False), "version": 2}


def _run_align(s):
    """Results and traces in task order (the arena holds the traces in the order the tasks finished)."""
    r = la_batch_device(s.tasks, tspace=s.case["tspace"])
    s.last = r   # the views below read its buffers
    res = torch.as_tensor(_View(r.results, 20 * r.n, "<i4"), device="cuda").view(r.n, 20)
    arena = torch.as_tensor(_View(r.arena, max(r.used, 1), "<i2"), device="cuda")
    n = (res[:, 10] + res[:, 11]).to(torch.int64)
    at = torch.where(n > 0, res[:, 12:14].contiguous().view(torch.int64).view(-1), 0)
    first = torch.cumsum(n, 0) - n
    idx = torch.arange(r.used, device="cuda") + torch.repeat_interleave(at - first, n, output_size=r.used)
    traces = torch.zeros(_trace_values(s.case), dtype=torch.int16, device="cuda")
    traces[:r.used] = arena[idx]
    return {"fields": torch.cat([res[:, :12], res[:, 16:]], 1), "traces": traces}


def _run_trace(s):
    c = s.case
    rc = lib.mi_trace_pts_host(100, c["mode"], s.packed.ctypes.data, s.packed.shape[0], s.points.ctypes.data,
                               s.points.shape[0], s.trace_tasks.ctypes.data_as(C.POINTER(MiTraceTask)), s.n,
                               s.results.ctypes.data_as(C.POINTER(MiTraceResult)), s.trace.ctypes.data,
                               s.trace.shape[0])
    if rc != 0:
        raise RuntimeError(f"mi_trace_pts_host failed ({rc}): {lib.last_error()}")
    return {"diffs": s.results["diffs"], "ntrace": s.results["ntrace"], "trace": s.trace}


def _run_dust(s):
    c = s.case
    rc = s.dal.h.mi_dust(C.byref(s.blocks[0]), c["window"], c["threshold"], c["mlen"], 0, s.anno.ctypes.data,
                         s.points.ctypes.data)
    if rc != 0:
        raise RuntimeError(f"mi_dust failed ({rc})")
    return {"anno": s.anno, "points": s.points[:s.npoints]}


def _run_lasort(s):
    n = C.c_longlong(0)
    rc = s.dal.h.mi_las_sort(s.body.ctypes.data, s.body.nbytes, s.n, 100, s.out.ctypes.data, C.byref(n))
    if rc != 0:
        raise RuntimeError(f"mi_las_sort failed ({rc})")
    return s.out


def run(state):
    return {"overlap": _run_overlap, "pair": _run_pair, "align": _run_align, "trace": _run_trace, "dust": _run_dust,
            "lasort": _run_lasort}[state.case["kind"]](state)


# ---- what a pass cannot do without ------------------------------------------------------


def work(case):
    """Bytes: the packed reads (2 bits a base) and every result once.  flops: integer operations of the furthest-
    reaching wave, whose band cells and snake steps no exact implementation leaves out (10 a cell, 2 a snake step):
    one wave per difference of an overlap, a band of 2 * 30 * err diagonals (the lag the waves are trimmed to over
    the advance a difference gives), and a snake step per cell and matched base."""
    k = case["kind"]

    def aligned(bases, pair_err):
        waves = bases * pair_err
        band = max(3.0, 60.0 * pair_err)
        return waves * band * (10 + 2 * (1 + 0.33 + 1.0 / (pair_err * band)))

    if k in ("overlap", "pair"):
        bases = case["genome"] * case["coverage"]
        # pairs of reads overlap over half of a read at the mean; every pair is found once and reported in both orders
        share = 0.5 if k == "overlap" else 0.25
        pairs = share * bases / case["mean"] * 2.0 * case["coverage"]
        over = pairs * 0.5 * case["mean"]
        nbytes = bases / 4 + 2 * (pairs * 40 + over / case["tspace"] * (2 if case["tspace"] <= 125 else 4))
        return {"bytes": nbytes, "flops": aligned(over, 2 * case["err"])}
    mean = _mean_len(case) if k in ("align", "trace") else 0.0
    if k == "align":
        n, e = case["tasks"], (case["emin"] + case["emax"]) / 2
        nbytes = n * (2 * mean / 4 + 56 + 80 + 4 * 2 * mean / case["tspace"])
        return {"bytes": nbytes, "flops": n * aligned(mean, e)}
    if k == "trace":
        n, e = case["tasks"], (case["emin"] + case["emax"]) / 2
        # O(NP) between trace points 100 bases apart: about (100 e)^2 cells a segment
        return {"bytes": n * (2 * mean / 4 + 4 * mean / 100 + 4 * mean * e),
                "flops": n * mean / 100 * (100 * e) ** 2 * 10}
    if k == "dust":
        bases = case["genome"] * case["coverage"]
        return {"bytes": bases, "flops": 14.0 * bases}
    n = case["records"]
    return {"bytes": 2.0 * n * (40 + 2 * case["mean"] / 100), "flops": 0}


def tolerance(case):
    """Alignments, traces, tracks and files are pinned bit for bit, whatever the sizes and types."""
    return "exact"


def exact(case, seed):
    """Integers and bytes only: no output has a 64-bit value to be compared with."""
    return None
