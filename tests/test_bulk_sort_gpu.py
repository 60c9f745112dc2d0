"""Builds that the radix passes sort, against the oracle: 32-bit ones on both
sides of the size up to which segments fit the LDS, 64-bit ones whose keys vary
in a few digits only (passes over constant digits are skipped), at the edges of
the passes' tiles; and dumps of a single run, with and without tombstones."""

import numpy as np
import pytest

from test_batch_sort_gpu import Pair, keys_of
from test_flix_gpu import FlixPair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1 << 21, (1 << 21) + 1, (1 << 21) + 8193])
@pytest.mark.parametrize("kind", ["full", "narrow", "hot"])
def test_builds_32(gd, orc, io, n, kind):
    rng = np.random.default_rng(n)
    p = Pair(gd, orc, io, 4, n)
    k = keys_of(rng, n, kind, 4)
    v = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    p.d.bulk_build(p.up(k), p.up(v), count=n)
    assert p.o.bulk_build(k, v) == 0
    p.check(rng)


@pytest.mark.parametrize("low,high", [(13, 0), (30, 0), (8, 40), (0, 56),
                                      (17, 63)])
def test_builds_64_of_few_digits(gd, orc, io, low, high):
    n = (1 << 20) + 8191
    rng = np.random.default_rng(low)
    p = Pair(gd, orc, io, 8, n)
    k = rng.integers(0, 1 << low, n, dtype=np.uint64)
    if high:
        k += rng.integers(0, 2, n, dtype=np.uint64) << np.uint64(high)
    v = rng.integers(0, 1 << 63, n, dtype=np.uint64)
    p.d.bulk_build(p.up(k), p.up(v), count=n)
    assert p.o.bulk_build(k, v) == 0
    p.check(rng)


@pytest.mark.parametrize("erase", [False, True])
def test_dump_of_one_run(gd, orc, io, erase):
    rng = np.random.default_rng(1)
    p = Pair(gd, orc, io, 4, 50000)
    k = keys_of(rng, 50000, "full", 4)
    e = (rng.random(len(k)) < (0.3 if erase else 0.0)).astype(np.uint8)
    p.d.apply_mixed(p.up(k), p.up(k), io.up(e, np.uint8), count=len(k))
    assert p.o.apply_mixed(k, k, e) == 0
    p.check(rng)
    p.check(rng)


# the passes' tiles and workgroups change at 600,000 keys; grouped lookups take
# a chained and a prefix pass
@pytest.mark.parametrize("kb", [4, 8])
@pytest.mark.parametrize("n", [599999, 600000, 8192 * 74, 8192 * 74 + 1])
def test_passes_of_an_index(gd, orc, io, kb, n):
    rng = np.random.default_rng(n)
    p = FlixPair(gd, orc, io, kb, 4, node_slots=32)
    k = keys_of(rng, n, "runs", kb)
    p.build(k)
    add = keys_of(rng, n, "full", kb)
    p.insert(add, np.arange(n, dtype=np.uint32))
    q = np.concatenate([rng.choice(add, n // 2),
                        keys_of(rng, n - n // 2, "full", kb)])
    assert np.array_equal(p.lookup(q), p.o.lookup(q))
    p.remove(rng.permutation(add)[: n // 2])
    p.check_all(rng, 0, 1 << 31)
