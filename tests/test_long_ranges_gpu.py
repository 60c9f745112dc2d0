"""Range sums and counts of long ranges, which the waves of a workgroup and,
for few queries, of a team of workgroups share, against prefix sums of the
oracle's contents, bit for bit: lengths at the edges of the thresholds and
chunks (in rows of one run and of several, with shadowed versions and
tombstones), skewed keys (directory buckets wider than a row window), many
long ranges at once, and both key widths."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Filled:
    """A dictionary of several runs (none merges) and its live contents."""

    def __init__(self, gd, orc, io, key_bytes, sizes, erase, skew, seed):
        rng = np.random.default_rng(seed)
        self.kb, self.io = key_bytes, io
        self.dt = np.uint32 if key_bytes == 4 else np.uint64
        cfg = dict(max_elements=1 << 21, batch_capacity=1 << 18)
        self.d = gd.GPULSMOpt(key_bytes=key_bytes, tuning={"max_runs": 12},
                              **cfg)
        o = orc.LsmOracle(key_bytes=key_bytes, **cfg)
        top = 1 << (32 if key_bytes == 4 else 63)
        for n in sizes:
            keys = rng.integers(0, top, n, dtype=np.uint64)
            if skew:  # most keys in a sliver of the key space
                near = rng.random(n) < 0.9
                keys[near] = top // 2 + keys[near] % np.uint64(1 << 18)
            keys = keys.astype(self.dt)
            vals = rng.integers(0, 1 << 63, n, dtype=np.uint64).astype(self.dt)
            gone = (rng.random(n) < erase).astype(np.uint8)
            if o.size():
                again = rng.random(n) < 0.3
                keys[again] = rng.choice(o.dump()[0], int(again.sum()))
            self.d.apply_mixed(self.up(keys), self.up(vals),
                               io.up(gone, np.uint8), count=n)
            assert o.apply_mixed(keys, vals, gone) == 0
        self.keys, vals = o.dump()
        with np.errstate(over="ignore"):
            self.sums = np.concatenate(
                [np.zeros(1, np.uint64),
                 np.cumsum(vals.astype(np.uint64), dtype=np.uint64)])

    def up(self, a):
        return self.io.up(np.asarray(a, self.dt), self.dt)

    def check(self, lo, hi):
        n = len(lo)
        a = np.searchsorted(self.keys, lo, side="left")
        z = np.maximum(np.searchsorted(self.keys, hi, side="right"), a)
        dlo, dhi = self.up(lo), self.up(hi)
        for call, want in ((self.d.range, self.sums[z] - self.sums[a]),
                           (self.d.range_count, z - a)):
            out = self.io.empty(n, self.kb)
            call(dlo, dhi, out, count=n)
            assert np.array_equal(self.io.down(out, n, self.dt),
                                  want.astype(self.dt))


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("sizes,erase,skew", [
    ([150000], 0.0, False),
    ([150000, 60000, 20000], 0.2, False),
    ([1 << 17, 1 << 16, 1 << 15, 1 << 14, 1 << 13, 1000, 10], 0.1, False),
    ([90000, 40000, 9000], 0.0, True),
])
def test_long_ranges(gd, orc, io, key_bytes, sizes, erase, skew):
    f = Filled(gd, orc, io, key_bytes, sizes, erase, skew, 77)
    rng = np.random.default_rng(3)
    m = len(f.keys)
    lens = [1, 2, 8, 9, 63, 64, 65, 255, 256, 257, 511, 512, 513, 700, 1023,
            1024, 1025, 2049, 4096, 8191, 8192, 8193, 20000, 65537, m - 1, m]
    lens = np.array([x for x in lens if x <= m] * 6)
    i = (rng.random(len(lens)) * (m - lens + 1)).astype(np.int64)
    lo, hi = f.keys[i].copy(), f.keys[i + lens - 1].copy()
    hi[:3], lo[:3] = f.keys[0], f.keys[-1]           # inverted
    lo[3:6], hi[3:6] = 0, np.iinfo(f.dt).max         # everything
    f.check(lo, hi)


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("n", [1, 3, 2047, 2049, 190000])
def test_only_long_ranges(gd, orc, io, key_bytes, n):
    """Every range long: one query, the most that get teams, one more, and
    rounds of long queries only; twice, as the teams' sums start from zero
    in each call."""
    f = Filled(gd, orc, io, key_bytes, [140000, 5000], 0.1, False, 5)
    rng = np.random.default_rng(4)
    for _ in range(2):
        i = rng.integers(0, len(f.keys) - 1500, n)
        f.check(f.keys[i], f.keys[i + rng.integers(1100, 1500, n)])
