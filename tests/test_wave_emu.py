"""The batched aligner's device code on the CPU (tests/wave_emu) against the
oracle: the kernels of marvel_amd/csrc/la_pack.hpp and la_batch_core.hpp
compiled by g++, one fiber per lane."""

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
from repeat_tasks import long_read_task

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or os.uname().machine != "x86_64",
                                reason="needs g++ on x86-64")


@pytest.fixture(scope="module", params=[False, True], ids=["", "garbage"])
def emu(request):
    """One library as built, one whose LDS holds garbage when a kernel starts."""
    os.environ.setdefault("MI_EMU_CUS", "1")
    emu_lib.build()
    return emu_lib.Lib(request.param)


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
