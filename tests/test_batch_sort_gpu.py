"""64-bit updates and builds (and the 32-bit ones that the segmented admission
does not take) against the oracle, bit for bit: batches of one LDS piece and
of a piece per top digit, at their edges, and batches whose most frequent digit
does not fit the LDS (radix passes), with keys in both halves of the key space,
repeated keys, and erases, whose flags ride in a key bit or are gathered."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def keys_of(rng, n, kind, key_bytes):
    bits = 8 * key_bytes
    top = (1 << bits) - 1
    if kind == "full":
        x = rng.integers(0, top, n, dtype=np.uint64, endpoint=True)
    elif kind == "narrow":    # the low 13 bits vary: every key repeats
        x = rng.integers(0, 1 << 13, n, dtype=np.uint64) + np.uint64(1 << 20)
    elif kind == "half":      # the top bit does not vary
        x = rng.integers(0, top >> 1, n, dtype=np.uint64)
    elif kind == "hot":       # a few keys make up most of the batch
        x = rng.integers(0, top, n, dtype=np.uint64, endpoint=True)
        hot = rng.random(n) < 0.8
        x[hot] = rng.choice(x[:5], int(hot.sum()))
    elif kind == "islands":   # two dense stretches far apart
        x = rng.integers(0, 3 * n, n, dtype=np.uint64)
        x[rng.random(n) < 0.5] += np.uint64(top // 3 * 2)
    elif kind == "runs":      # stretches of consecutive keys
        s = rng.integers(0, top - 5000, max(1, n >> 11), dtype=np.uint64)
        x = rng.choice(s, n) + rng.integers(0, 4096, n, dtype=np.uint64)
    elif kind == "one":
        x = np.full(n, top // 5, np.uint64)
    else:                     # ascending
        x = np.arange(n, dtype=np.uint64) * np.uint64(3)
    return x.astype(np.uint32 if key_bytes == 4 else np.uint64)


KINDS = ["full", "narrow", "half", "hot", "islands", "runs", "one", "ascending"]


class Pair:
    def __init__(self, gd, orc, io, key_bytes, n):
        self.io, self.kb = io, key_bytes
        self.dt = np.uint32 if key_bytes == 4 else np.uint64
        cfg = dict(max_elements=4 * n + 1024, batch_capacity=1 << 20)
        self.d = gd.GPULSMOpt(key_bytes=key_bytes, **cfg)
        self.o = orc.LsmOracle(key_bytes=key_bytes, **cfg)

    def up(self, a):
        return self.io.up(np.asarray(a, self.dt), self.dt)

    def check(self, rng):
        ek, ev = self.o.dump()
        n = len(ek)
        ok, ov = self.io.empty(n + 1, self.kb), self.io.empty(n + 1, self.kb)
        assert self.d.dump_sorted(ok, ov, capacity=n + 1) == n
        assert np.array_equal(self.io.down(ok, n, self.dt), ek)
        assert np.array_equal(self.io.down(ov, n, self.dt), ev)
        # the directory: lookups and successors of stored and other keys
        top = np.iinfo(self.dt).max
        q = rng.integers(0, top, 20000, dtype=np.uint64,
                         endpoint=True).astype(self.dt)
        if n:
            q[:10000] = rng.choice(ek, 10000)
            q[10000:15000] = rng.choice(ek, 5000) + self.dt(1)
        for call, want in ((self.d.lookup, self.o.lookup(q)),
                           (self.d.successor, self.o.successor(q))):
            out = self.io.empty(len(q), self.kb)
            call(self.up(q), out, count=len(q))
            assert np.array_equal(self.io.down(out, len(q), self.dt), want)


SIZES64 = [2049, 6143, 6144, 6145, 9217, 30011, 100003, 700001, 1 << 20]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", SIZES64)
def test_batches_64(gd, orc, io, kind, n):
    rng = np.random.default_rng(n)
    p = Pair(gd, orc, io, 8, n)
    k = keys_of(rng, n, kind, 8)
    v = rng.integers(0, 1 << 63, n, dtype=np.uint64)
    e = (rng.random(n) < 0.25).astype(np.uint8)
    mode = (n + KINDS.index(kind)) % 3
    if mode == 0:
        p.d.insert(p.up(k), p.up(v), count=n)
        assert p.o.insert(k, v) == 0
    else:
        p.d.apply_mixed(p.up(k), p.up(v), io.up(e, np.uint8), count=n)
        assert p.o.apply_mixed(k, v, e) == 0
    p.check(rng)
    if mode == 2:  # tombstones of half of the keys
        gone = rng.permutation(k)[: max(1, n // 2)]
        p.d.erase(p.up(gone), count=len(gone))
        assert p.o.erase(gone) == 0
        p.check(rng)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("key_bytes,n", [(4, 5000), (4, 8193), (4, 1100000),
                                         (8, 1048577)])
def test_builds(gd, orc, io, kind, key_bytes, n):
    rng = np.random.default_rng(7)
    p = Pair(gd, orc, io, key_bytes, n)
    k = keys_of(rng, n, kind, key_bytes)
    v = rng.integers(0, 1 << 63, n, dtype=np.uint64).astype(p.dt)
    p.d.bulk_build(p.up(k), p.up(v), count=n)
    assert p.o.bulk_build(k, v) == 0
    p.check(rng)
