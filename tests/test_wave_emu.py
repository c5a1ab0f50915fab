"""The batched aligner's device code on the CPU (tests/wave_emu) against the
oracle: the kernels of marvel_amd/csrc/la_pack.hpp and la_batch_core.hpp
compiled by g++, one fiber per lane."""

import ctypes as C
import os
import shutil

import numpy as np
import pytest

import emu_lib
import la_golden
import oracle_lib
import repeat_tasks
from marvel_amd import latasks
from marvel_amd.align import la_batch
from marvel_amd.lib import MiLaResult, MiLaTask, MiTuning, params
from repeat_tasks import long_read_task

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or os.uname().machine != "x86_64",
                                reason="needs g++ on x86-64")


@pytest.fixture(scope="module", params=[False, True], ids=["", "garbage"])
def emu(request):
    """One library as built, one whose LDS holds garbage when a kernel starts.
    On one CU with 4 waves, so that batches of more than 4 tasks use both halves of a wave."""
    os.environ["MI_EMU_CUS"] = "1"
    emu_lib.build()
    lib = emu_lib.Lib(request.param)
    assert lib.mi_set_tuning(C.byref(MiTuning(0, 0, 0, 4, 0))) == 0
    return lib


def check(emu, ts):
    """Every task the oracle defines is its result, every other one status 3; returns the number of the former."""
    want, st = oracle_lib.run_tasks(ts)
    with emu_lib.in_place_of_gpu(emu):
        got, status = la_batch(ts)
    keep = [i for i in range(ts.n) if st[i] == 0]
    bad = la_golden.diff([got[i] for i in keep], [want[i] for i in keep], status[keep])
    assert not bad, "\n".join(bad)
    assert all(status[i] == 3 for i in range(ts.n) if st[i] != 0)
    return len(keep)


@pytest.mark.parametrize("tspace,offmax,emax", [(100, 5, 0.25), (100, 60, 0.25), (100, 200, 0.2), (126, 5, 0.12),
                                                (13, 5, 0.12)])
def test_noisy_pairs(emu, tspace, offmax, emax):
    assert check(emu, latasks.make_tasks(20, tspace + offmax, lmin=300, lmax=2500, emin=0.02, emax=emax,
                                         offmax=offmax, tspace=tspace)) >= 14


def test_one_task_leaves_half_the_wave_idle(emu):
    check(emu, latasks.make_tasks(1, 5, lmin=800, lmax=1500, emin=0.1, emax=0.2, offmax=0))


@pytest.mark.parametrize("width", [2, 30, 31, 90])
def test_initial_bands(emu, width):
    ts = latasks.make_tasks(6, 300 + width, lmin=1500, lmax=2500, emin=0.05, emax=0.15, offmax=0)
    par = ts.par.copy()
    par[:, 3] -= width // 2
    par[:, 4] = par[:, 3] + width - 1
    check(emu, latasks.TaskSet(ts.ave_corr, ts.tspace, ts.freq, ts.reads, par.astype(np.int32)))


@pytest.mark.parametrize("tspace", [5, 20, 100])
@pytest.mark.parametrize("width,points,tail", [(1, (250, 420), 0), (5, (128, 260), 0), (5, (260, 420), 2500),
                                               (20, (128, 260), 2500), (40, (260, 420), 0), (150, (128, 300), 0)])
def test_exact_tandem_repeats(emu, tspace, width, points, tail):
    """Paths more than 128 and more than 256 trace points ahead of a
    diagonal's thresholds: a pebble's point is known by 8 bits of its number
    (far_points, la_pack.hpp)."""
    check(emu, repeat_tasks.make(6, 1000 * tspace + width + tail, tspace, points, width=width, tail=tail))


@pytest.mark.parametrize("tspace", [2**23 - 1, 2**23, 9_000_000, 2**30])
def test_trace_spacings_beyond_24_bits(emu, tspace):
    """Trace points are placed by 24-bit products (point_at, la_pack.hpp)."""
    assert check(emu, latasks.make_tasks(8, 5, lmin=300, lmax=900, emin=0.02, emax=0.2, offmax=20, tspace=tspace)) == 8


@pytest.mark.parametrize("tspace", [1, 2, 100, 2**23, 2**24])
def test_a_read_of_more_than_2_to_23_bases(emu, tspace):
    assert check(emu, long_read_task(tspace)) == 1


def wide_task(width, length=3000, tspace=100):
    """One task that starts on `width` diagonals."""
    ts = latasks.make_tasks(1, 7, lmin=length, lmax=length + 1, emin=0.05, emax=0.1, offmax=0, tspace=tspace)
    par = ts.par.copy()
    par[:, 3] -= width // 2
    par[:, 4] = par[:, 3] + width - 1
    return latasks.TaskSet(ts.ave_corr, ts.tspace, ts.freq, ts.reads, par)


def test_a_single_task_beyond_the_widest_window(emu):
    """The workspace of a batch of one holds the last level's scratch; the task keeps status 1 (window)."""
    with emu_lib.in_place_of_gpu(emu):
        assert la_batch(wide_task(1100))[1].tolist() == [1]


def noalloc(emu, ts):
    """mi_la_batch_device_noalloc over a TaskSet (device memory is host memory here): (rc, status, results, traces)."""
    words, aw, bw = ts.packed()
    tasks, res = (MiLaTask * ts.n)(), (MiLaResult * ts.n)()
    for i in range(ts.n):
        t = tasks[i]
        t.aword, t.bword = int(aw[i]), int(bw[i])
        t.alen, t.blen, t.comp, t.low, t.hgh, t.anti, t.lbord, t.hbord = (int(x) for x in ts.par[i])
    cap = int(sum(4 * (max(int(p[0]), int(p[1])) // ts.tspace + 2) for p in ts.par)) + 16
    tr, used = np.zeros(cap, dtype=np.uint16), C.c_ulonglong(0)
    prm = params(ts.ave_corr, ts.tspace, ts.freq)
    rc = emu.mi_la_batch_device_noalloc(C.byref(prm), words.ctypes.data, words.shape[0], tasks, ts.n, res,
                                        tr.ctypes.data, cap, C.byref(used))
    out = [((r.abpos, r.bbpos, r.aepos, r.bepos, r.diffs, r.atlen, r.b_abpos, r.b_bbpos, r.b_aepos, r.b_bepos, r.diffs,
             r.btlen), tr[r.atrace:r.atrace + r.atlen], tr[r.btrace:r.btrace + r.btlen]) for r in res]
    return rc, np.array([r.status for r in res]), out


@pytest.mark.parametrize("n", [1, 130])
def test_fixed_scratch_batch(emu, n):
    """130: more tasks than the 64 MiB hold waves."""
    ts = latasks.make_tasks(n, 12, lmin=200, lmax=400, emin=0.05, emax=0.2, offmax=10)
    want, st = oracle_lib.run_tasks(ts)
    rc, status, got = noalloc(emu, ts)
    keep = [i for i in range(n) if st[i] == 0]
    assert rc == 0 and len(keep) > 0.9 * n
    assert not la_golden.diff([got[i] for i in keep], [want[i] for i in keep], status[keep])


def test_fixed_scratch_holds_one_wave_of_the_last_level(emu):
    """A read of 500,000 bases at a spacing of 1: the last level's pool, chain
    points and traces fit into 64 MiB once, not twice."""
    ts = wide_task(1100, tspace=1)
    long = np.concatenate([ts.reads[0], np.zeros(500_000 - len(ts.reads[0]), dtype=np.uint8)])
    par = ts.par.copy()
    par[0, 0] = len(long)
    rc, status, _ = noalloc(emu, latasks.TaskSet(ts.ave_corr, 1, ts.freq, [long, ts.reads[1]], par))
    assert rc == 0 and status.tolist() == [1]
