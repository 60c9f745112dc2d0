"""Ranges over four or more runs, whose rows are resolved in LDS (a wave's
together up to 512 rows, a workgroup's up to 2048), against prefix sums of the
oracle's contents: rows at the edges of both, of several versions and
tombstones, dense and spread keys, one query and many per wave, and through the
serving engine's fused steps."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Runs:
    """Batches that stay runs of their own, and their live contents."""

    def __init__(self, orc, io, key_bytes, runs, rows, dense, seed):
        rng = np.random.default_rng(seed)
        self.kb, self.io = key_bytes, io
        self.dt = np.uint32 if key_bytes == 4 else np.uint64
        top = 3 * rows if dense else np.iinfo(self.dt).max
        o = orc.LsmOracle(key_bytes=key_bytes, max_elements=1 << 20,
                          batch_capacity=1 << 18)
        self.batches, every = [], []
        for i in range(runs):
            n = rows - i * (rows // (2 * runs))  # falling: none merges
            k = rng.integers(0, top, n, dtype=np.uint64, endpoint=True)
            if every:
                again = rng.random(n) < 0.4
                k[again] = rng.choice(np.concatenate(every), int(again.sum()))
            k = k.astype(self.dt)
            v = rng.integers(0, 1 << 63, n, dtype=np.uint64).astype(self.dt)
            gone = (rng.random(n) < 0.2).astype(np.uint8)
            self.batches.append((k, v, gone))
            assert o.apply_mixed(k, v, gone) == 0
            every.append(np.unique(k))
        self.rows = np.sort(np.concatenate(every))  # every version
        self.keys, vals = o.dump()
        with np.errstate(over="ignore"):
            self.sums = np.concatenate(
                [np.zeros(1, np.uint64),
                 np.cumsum(vals.astype(np.uint64), dtype=np.uint64)])

    def up(self, a):
        return self.io.up(np.asarray(a, self.dt), self.dt)

    def fill(self, d):
        for k, v, gone in self.batches:
            d.apply_mixed(self.up(k), self.up(v), self.io.up(gone, np.uint8),
                          count=len(k))

    def ranges(self, rng, lengths):
        """A range of about so many rows for each of the lengths."""
        lengths = np.minimum(lengths, len(self.rows))
        i = (rng.random(len(lengths)) *
             (len(self.rows) - lengths + 1)).astype(np.int64)
        return self.rows[i], self.rows[i + lengths - 1]

    def want(self, lo, hi, count):
        a = np.searchsorted(self.keys, lo, side="left")
        z = np.maximum(np.searchsorted(self.keys, hi, side="right"), a)
        return (z - a if count else self.sums[z] - self.sums[a]).astype(self.dt)

    def check(self, d, lo, hi):
        for call, count in ((d.range, False), (d.range_count, True)):
            out = self.io.empty(len(lo), self.kb)
            call(self.up(lo), self.up(hi), out, count=len(lo))
            assert np.array_equal(self.io.down(out, len(lo), self.dt),
                                  self.want(lo, hi, count))


def edges():
    near = [x + d for x in (1, 64, 256, 512, 1024, 2048, 2600)
            for d in range(-9, 10)]
    return np.array([x for x in near if x > 0], np.int64)


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("runs,rows", [(3, 9000), (4, 9000), (5, 70000),
                                       (10, 3000), (40, 400)])
@pytest.mark.parametrize("dense", [False, True])
def test_ranges_over_many_runs(gd, orc, io, key_bytes, runs, rows, dense):
    f = Runs(orc, io, key_bytes, runs, rows, dense, runs)
    d = gd.GPULSMOpt(key_bytes=key_bytes, max_elements=1 << 20,
                     batch_capacity=1 << 18,
                     tuning={"max_runs": 47, "merge_ways": 2})
    f.fill(d)
    assert d.shape()[0] == runs
    rng = np.random.default_rng(runs)
    lo, hi = f.ranges(rng, np.tile(edges(), 4))
    lo[:5], hi[:5] = hi[:5].copy(), lo[:5].copy()
    lo[5], hi[5] = 0, np.iinfo(f.dt).max
    f.check(d, lo, hi)
    f.check(d, lo[-1:], hi[-1:])                # a query on its own
    for longest in (12, 120, 700):              # several per wave
        lo, hi = f.ranges(rng, rng.integers(1, longest, 7001))
        f.check(d, lo, hi)
    assert d.shape()[0] == runs                 # (no call merged them)


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("step_launch", ["kernels", "direct", "graph"])
def test_serving_over_many_runs(gd, orc, io, key_bytes, step_launch):
    import torch
    f = Runs(orc, io, key_bytes, 8, 4000, False, 3)
    s = gd.Server(key_bytes=key_bytes, max_elements=1 << 20,
                  batch_capacity=1 << 18, step_launch=step_launch,
                  tuning={"max_runs": 47, "merge_ways": 2})
    for k, v, gone in f.batches:
        new, old = np.flatnonzero(gone == 0), np.flatnonzero(gone)
        # (the last update of a key wins: one request holds both kinds' order)
        last = {int(x): i for i, x in enumerate(k)}
        new = np.array([i for i in new if last[int(k[i])] == i], np.int64)
        old = np.array([i for i in old if last[int(k[i])] == i], np.int64)
        a, b, c = f.up(k[new]), f.up(v[new]), f.up(k[old])
        torch.cuda.synchronize()
        s.wait(s.submit(s.INSERT, a, b, count=len(new)))
        s.wait(s.submit(s.ERASE, c, count=len(old)))
    rng = np.random.default_rng(9)
    for n, longest in ((1, 60), (33, 60), (70, 3000)):
        lo, hi = f.ranges(rng, rng.integers(1, longest, n))
        dlo, dhi = f.up(lo), f.up(hi)
        for op, count in ((s.RANGE_SUM, False), (s.RANGE_COUNT, True)):
            out = io.empty(n, key_bytes)
            torch.cuda.synchronize()
            s.wait(s.submit(op, dlo, dhi, out, count=n))
            assert np.array_equal(io.down(out, n, f.dt), f.want(lo, hi, count))
    s.close()
