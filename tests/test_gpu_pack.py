"""The packed aligner (two alignments per wave, marvel_amd/csrc/la_pack.hpp)
at the sizes where its paths change, against the oracle: batches that leave
the upper halves idle and batches that use them, bands that stay within a
half's 30 diagonals, that outgrow them for a while, and that outgrow the 128
diagonals of the first wide window; trace spacings below and above the snake
step, whose trace-point numbers wrap at 256; initial bands of several
diagonals up to and beyond a half; exact tandem repeats, in which a path gets
more than 128 or 256 trace points ahead of a diagonal that takes it; and
trace points whose spacing or number is beyond 23 bits."""

import numpy as np
import pytest

import la_golden
import oracle_lib
import repeat_tasks
from marvel_amd import latasks
from marvel_amd.align import la_batch
from marvel_amd.lib import MiTuning, lib

pytestmark = pytest.mark.gpu


def _check(ts):
    want, st = oracle_lib.run_tasks(ts)
    got, status = la_batch(ts)
    keep = [i for i in range(ts.n) if st[i] == 0]
    bad = la_golden.diff([got[i] for i in keep], [want[i] for i in keep], status[keep])
    assert not bad, "\n".join(bad)
    assert all(status[i] == 3 for i in range(ts.n) if st[i] != 0)
    return len(keep)


@pytest.fixture
def few_waves():
    """1,024 waves on 256 CUs: batches beyond that use both halves of a wave."""
    import ctypes as C
    t = MiTuning(0, 0, 0, 4, 0)
    assert lib.mi_set_tuning(C.byref(t)) == 0
    yield
    lib.mi_set_tuning(None)


@pytest.mark.parametrize("offmax", [0, 15, 40, 200])
@pytest.mark.parametrize("tspace", [7, 100, 250])
def test_bands_and_trace_spacings(tspace, offmax):
    ts = latasks.make_tasks(48, 900 + offmax + tspace, lmin=300, lmax=4000, emin=0.02, emax=0.25, offmax=offmax,
                            tspace=tspace)
    print(f"[pack] tspace={tspace} offmax={offmax} n={ts.n}", flush=True)
    assert _check(ts) >= 40


@pytest.mark.parametrize("n", [1, 2, 1024, 1025, 2600])
def test_one_and_two_alignments_per_wave(n, few_waves):
    ts = latasks.make_tasks(n, 77 + n, lmin=200, lmax=700, emin=0.05, emax=0.25, offmax=30)
    print(f"[pack] n={n}", flush=True)
    _check(ts)


@pytest.mark.parametrize("width", [2, 29, 30, 31, 90, 200])
def test_initial_bands(width):
    """Local_Alignment started on `width` diagonals around the seed's."""
    ts = latasks.make_tasks(12, 300 + width, lmin=1500, lmax=3000, emin=0.05, emax=0.15, offmax=0)
    par = ts.par.copy()
    keep = []
    for i in range(ts.n):
        low = int(par[i, 3]) - width // 2
        hgh = low + width - 1
        alen, blen, anti = int(par[i, 0]), int(par[i, 1]), int(par[i, 5])
        # every start point inside both reads
        if all(0 <= (anti - k) // 2 <= blen and 0 <= (anti - k) // 2 + k <= alen for k in (low, hgh)):
            par[i, 3], par[i, 4] = low, hgh
            keep.append(i)
    assert len(keep) >= 4
    reads = [r for i in keep for r in (ts.reads[2 * i], ts.reads[2 * i + 1])]
    print(f"[pack] width={width} n={len(keep)}", flush=True)
    _check(latasks.TaskSet(ts.ave_corr, ts.tspace, ts.freq, reads, par[np.array(keep)]))


@pytest.mark.parametrize("tspace", [10, 20, 50, 100])
@pytest.mark.parametrize("width,tail", [(1, 0), (2, 2500), (5, 0), (20, 2500), (40, 0), (150, 2500)])
def test_exact_tandem_repeats(tspace, width, tail):
    for points in ((128, 260), (260, 420)):
        ts = repeat_tasks.make(16, 31 * tspace + width + points[0], tspace, points, width=width, tail=tail)
        print(f"[pack] repeats tspace={tspace} width={width} points={points} tail={tail}", flush=True)
        _check(ts)


def test_exact_tandem_repeats_on_both_halves(few_waves):
    ts = repeat_tasks.make(1400, 8, 10, (128, 300), width=5, tail=200, flank=100)
    print(f"[pack] repeats n={ts.n}", flush=True)
    _check(ts)


@pytest.mark.parametrize("tspace", [2**23 - 1, 2**23, 9_000_000, 2**30])
def test_trace_spacings_beyond_24_bits(tspace):
    ts = latasks.make_tasks(8, 5, lmin=300, lmax=900, emin=0.02, emax=0.2, offmax=20, tspace=tspace)
    print(f"[pack] tspace={tspace}", flush=True)
    assert _check(ts) == 8


@pytest.mark.parametrize("tspace", [1, 100, 2**24])
def test_a_read_of_more_than_2_to_23_bases(tspace):
    print(f"[pack] long read, tspace={tspace}", flush=True)
    assert _check(repeat_tasks.long_read_task(tspace)) == 1
