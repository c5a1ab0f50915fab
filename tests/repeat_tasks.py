"""Local_Alignment tasks over long exact tandem repeats, and over a very long
read.

Inside an exact repeat of a short period some diagonals of a band run to its
end in one wave while the ones between them stay where they are, so a
diagonal can inherit, one wave later, a path that is hundreds of trace points
ahead of its own thresholds."""

from __future__ import annotations

import numpy as np

from marvel_amd import latasks, sim


def make(n: int, seed: int, tspace: int, points, err=(0.02, 0.25), width: int = 1, tail: int = 0, flank: int = 600,
         periods=range(2, 12), ave_corr: float = 0.70, comp=None) -> latasks.TaskSet:
    """n tasks whose reads hold an exact tandem repeat of points[0] to
    points[1] trace spacings between two noisy flanks, with `tail` unrelated
    bases at each end.  The repeats of the two reads differ by up to one
    period, the seed lies in the left flank, on its border or inside, on
    `width` diagonals around its own (widths that leave a read are cut)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    reads, par = [], np.zeros((n, 8), dtype=np.int32)
    rand = lambda m: rng.integers(0, 4, size=m, dtype=np.uint8)
    for i in range(n):
        per = int(rng.choice(list(periods)))
        unit = rand(per)
        while len(set(unit.tolist())) == 1:
            unit = rand(per)
        rep = int(rng.integers(points[0] * tspace, points[1] * tspace))
        e = rng.uniform(*err) / 2
        fl, fr = rand(flank), rand(flank)
        side, seed_at = [], int(rng.integers(0, 3))
        p = int(rng.integers(flank // 4, flank))
        for _ in range(2):
            l, lm = latasks.mutate_map(fl, rng, e * 9 / 15, e * 4 / 15, e * 2 / 15)
            r, _m = latasks.mutate_map(fr, rng, e * 9 / 15, e * 4 / 15, e * 2 / 15)
            m = np.tile(unit, rep // per + 2)[:rep + int(rng.integers(0, per + 1))]
            at = tail + (int(lm[p]) if seed_at == 0 else len(l) if seed_at == 1 else len(l) + rep // 2)
            side.append((np.concatenate([rand(tail), l, m, r, rand(tail)]).astype(np.uint8), at))
        (a, x), (b, y) = side
        reads += [a, b]
        low = x - y - width // 2
        hgh = low + width - 1
        ok = [k for k in range(low, hgh + 1) if 0 <= (x + y - k) >> 1 <= len(b) and 0 <= ((x + y - k) >> 1) + k <= len(a)]
        par[i] = (len(a), len(b), int(rng.integers(0, 2)) if comp is None else comp, ok[0], ok[-1], x + y, -1, -1)
    return latasks.TaskSet(ave_corr, tspace, (0.25, 0.25, 0.25, 0.25), reads, par)


def reads(seed: int, tspace: int, error: float, coverage: float = 8.0, length: int = 6000):
    """Reads of a genome of exact tandem repeats (130 to 300 trace spacings
    long, periods 2 to 7) between stretches without."""
    g = sim.random_genome(length, seed)
    rng = np.random.default_rng(seed)
    at = 700
    while at + tspace * 260 < length:
        per = int(rng.integers(2, 8))
        unit = rng.integers(0, 4, per, dtype=np.uint8)
        ln = min(int(rng.integers(tspace * 130, tspace * 300)), length - at)
        g[at:at + ln] = np.tile(unit, ln // per + 1)[:ln]
        at += ln + int(rng.integers(500, 900))
    return sim.simulate_reads(g, coverage, 3500.0, 800.0, 2000, seed + 1, p_ins=error * .6, p_del=error * .27,
                              p_sub=error * .13).reads


def long_read_task(tspace: int) -> latasks.TaskSet:
    """A short read against the end of one of 2^23 + 3,000 bases: the numbers
    of the trace points around the seed are beyond 23 bits at a spacing of 1."""
    rng = np.random.Generator(np.random.PCG64(4))
    t = rng.integers(0, 4, 1500, dtype=np.uint8)
    a, am = latasks.mutate_map(t, rng, 0.03, 0.013, 0.007)
    b, bm = latasks.mutate_map(t, rng, 0.03, 0.013, 0.007)
    at = 2**23 + 3000 - len(a) - 100
    read = np.concatenate([rng.integers(0, 4, at, dtype=np.uint8), a, rng.integers(0, 4, 100, dtype=np.uint8)])
    x, y = at + int(am[700]), int(bm[700])
    return latasks.TaskSet(0.70, tspace, (0.25, 0.25, 0.25, 0.25), [read, b],
                           np.array([[len(read), len(b), 0, x - y, x - y, x + y, -1, -1]], dtype=np.int32))
