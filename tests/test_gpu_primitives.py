"""Wave64 building blocks of the aligner and the trace kernel on the GPU against CPU semantics."""

import numpy as np
import pytest

from marvel_amd import latasks
from marvel_amd.lib import lib

pytestmark = pytest.mark.gpu


def _run(which, inp=None, inp2=None, q=None, arg=0, nout=0):
    out = np.zeros(nout, dtype=np.int32)
    a = inp if inp is not None else np.zeros(1, dtype=np.int32)
    b = inp2 if inp2 is not None else np.zeros(1, dtype=np.int32)
    qq = q if q is not None else np.zeros((1, 4), dtype=np.int32)
    rc = lib.mi_selftest(which, a.ctypes.data, a.nbytes if inp is not None else 0, b.ctypes.data,
                         b.nbytes if inp2 is not None else 0, qq.ctypes.data, qq.shape[0] if q is not None else 0,
                         arg, out.ctypes.data, out.nbytes)
    assert rc == 0, lib.last_error()
    return out


def test_persistent_loop():
    print("[prim] persistent", flush=True)
    out = _run(0, arg=37, nout=5000)
    assert np.array_equal(out, 3 * np.arange(5000) + 1)


def test_lane_ops():
    print("[prim] lanes", flush=True)
    rng = np.random.default_rng(5)
    waves = 64
    v = rng.integers(0, 1000, size=waves * 64).astype(np.int32)
    out = _run(1, inp=v, arg=990, nout=waves * 64 * 8).reshape(waves, 64, 8)
    for w in range(waves):
        x = v[w * 64:(w + 1) * 64]
        for ln in range(64):
            o = out[w, ln]
            assert o[0] == (x[ln + 1:].max() if ln < 63 else -1)
            assert o[1] == (x[:ln].min() if ln > 0 else 2**31 - 1)
            assert o[2] == x[(ln - 1) % 64] and o[3] == x[(ln + 1) % 64]
            odd = np.nonzero(x & 1)[0]
            assert o[4] == (x[odd[0]] if len(odd) else -7)
            assert o[5] == int(((x[:ln] & 1) != 0).sum())
            assert o[6] == int((x > 990).any())
            assert o[7] == len(odd)


def test_trace_matchers():
    """match_fwd / match_rev, the trace kernel's."""
    print("[prim] matchers", flush=True)
    rng = np.random.default_rng(9)
    L = 3000
    a = rng.integers(0, 4, size=L, dtype=np.uint8)
    b = a.copy()
    flip = rng.random(L) < 0.05
    b[flip] = (b[flip] + 1) & 3
    wa, oa = latasks.pack_reads([a])
    wb, ob = latasks.pack_reads([b])
    assert oa[0] == 1 and ob[0] == 1
    qs = []
    for _ in range(4000):
        d = int(rng.integers(0, 2)) * 2 - 1
        x = int(rng.integers(0, L + 1))
        y = x
        lim = (L - x) if d > 0 else x
        lim = int(rng.integers(0, lim + 1))
        qs.append((x, y, lim, d))
    q = np.array(qs, dtype=np.int32)
    out = _run(2, inp=wa, inp2=wb, q=q, nout=2 * len(qs)).reshape(-1, 2)
    for i, (x, y, lim, d) in enumerate(qs):
        s = 0
        if d > 0:
            while s < lim and a[x + s] == b[y + s]:
                s += 1
        else:
            while s < lim and a[x - 1 - s] == b[y - 1 - s]:
                s += 1
        assert out[i, 0] == s and out[i, 1] == int(s < lim), (i, x, y, lim, d, out[i], s)


def test_lane_moves():
    """The aligner's scans, neighbour moves and gathers, at the ends of the halves and of the wave too."""
    print("[prim] moves", flush=True)
    rng = np.random.default_rng(9)
    waves = 8
    sent = -(1 << 30)
    v = rng.integers(-2**30, 2**30, size=waves * 64).astype(np.int32)
    v[64:128] = np.arange(64, dtype=np.int32)            # increasing
    v[128:192] = np.arange(64, 0, -1, dtype=np.int32)    # decreasing
    v[192:256] = 7                                       # constant
    v[256:320] = sent                                    # all sentinels
    v[320::5] = sent                                     # scattered sentinels
    out = _run(3, inp=v, nout=waves * 64 * 13).reshape(waves, 64, 13)
    lanes = np.arange(64)
    for w in range(waves):
        x, o = v[w * 64:(w + 1) * 64], out[w]
        assert np.array_equal(o[:32, 0], np.maximum.accumulate(x[:32]))
        assert np.array_equal(o[32:, 0], np.maximum.accumulate(x[32:]))
        assert np.array_equal(o[:, 1], np.maximum.accumulate(x))
        assert np.array_equal(o[1:, 2], x[:-1])          # (lane 0: anything)
        assert np.array_equal(o[:-1, 3], x[1:])          # (lane 63: anything)
        assert np.array_equal(o[:, 4], np.insert(x[:-1], 0, sent))
        assert np.array_equal(o[:, 5], np.append(x[1:], sent))
        assert np.array_equal(o[:, 6], x[(7 * lanes + 3) & 63])
        assert np.array_equal(o[:, 7], x[lanes ^ 33]) and np.array_equal(o[:, 8], ~x[lanes ^ 33])
        odd = x & 1
        assert np.array_equal(o[:, 9], odd)
        for h in (0, 1):
            bits = odd[32 * h:32 * h + 32]
            mask = int((bits.astype(np.uint64) << np.arange(32, dtype=np.uint64)).sum())
            at = np.flatnonzero(bits)
            want = (mask, at[-1] if len(at) else -1, at[0] if len(at) else -1)
            for ln in range(32 * h, 32 * h + 32):
                assert (int(o[ln, 10]) & 0xffffffff, int(o[ln, 11]), int(o[ln, 12])) == want


def test_snake_of_32_bases_a_step():
    """snake_len forward and reverse: limits around its step, runs of many
    steps, windows that begin in the guard word before a read or end in those
    after it, lanes without a query."""
    print("[prim] snake_len", flush=True)
    rng = np.random.default_rng(10)
    L = 2011
    a = rng.integers(0, 4, size=L, dtype=np.uint8)
    b = a.copy()
    flip = rng.random(L) < 0.04
    flip[:40] = flip[600:1100] = flip[-40:] = False   # runs of 0, 1 and more than 10 steps
    b[flip] = (b[flip] + 1) & 3
    wa, _ = latasks.pack_reads([a])
    wb, _ = latasks.pack_reads([b])
    qs, want = [], []
    for i in range(3001):
        m = -int(rng.integers(0, 2))
        x = int(rng.integers(0, L + 1)) if i % 4 else int(rng.choice([0, 1, 31, 32, 33, L - 33, L - 32, L - 1, L]))
        room = L - x if m == 0 else x
        lim = min(room, int(rng.choice([0, 1, 31, 32, 33, 63, 64, 65, room])))
        s = 0
        if m == 0:
            while s < lim and a[x + s] == b[x + s]:
                s += 1
        else:
            while s < lim and a[x - 1 - s] == b[x - 1 - s]:
                s += 1
        qs.append((x, x, lim, m) if m == 0 else (-x, -x, lim, m))
        want.append(s)
    out = _run(4, inp=wa, inp2=wb, q=np.array(qs, dtype=np.int32), nout=len(qs))
    bad = [(qs[i], want[i], int(out[i])) for i in range(len(qs)) if out[i] != want[i]]
    assert not bad, bad[:5]


def test_path_columns():
    """add_columns and min_suffix against a list of a path's columns: every
    step is a mismatch and then s matches; a path begins as a mismatch and 60
    matches."""
    import ctypes as C

    from marvel_amd.lib import params

    print("[prim] columns", flush=True)
    rng = np.random.default_rng(11)
    waves, steps = 4, 40
    s = rng.choice([0, 1, 2, 3, 5, 9, 10, 29, 30, 31, 59, 60, 61, 62, 500], size=(waves * 64, steps),
                   p=[.25, .2, .15, .1, .05, .05, .04, .03, .02, .02, .02, .02, .02, .02, .01]).astype(np.int32)
    out = _run(5, inp=s, arg=steps, nout=waves * 64 * steps * 2).reshape(waves * 64, steps, 2)
    ave, ms, ds = C.c_int(), C.c_int(), C.c_int()
    prm = params(0.70, 100, (0.25,) * 4)
    assert lib.mi_align_params(C.byref(prm), C.byref(ave), C.byref(ms), C.byref(ds)) == 0
    for i in range(0, waves * 64, 3):
        cols = [0] + [1] * 60
        for t in range(steps):
            cols += [0] + [1] * int(s[i, t])
            del cols[:-61]
            suffix = np.cumsum([ms.value if c else -ds.value for c in cols[:-31:-1]])
            assert tuple(out[i, t]) == (sum(cols), suffix.min()), (i, t)
