"""Successors whose neighbouring queries pass different numbers of dead keys,
held by one run or by several, against the oracle; and of a dictionary without
rows."""

import numpy as np
import pytest

from test_batch_sort_gpu import Pair

pytestmark = pytest.mark.gpu


def successors(p, io, key_bytes, q):
    out = io.empty(len(q), key_bytes)
    p.d.successor(p.up(q), out, count=len(q))
    return io.down(out, len(q), p.dt)


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("runs", [2, 3, 7, 9])
def test_uneven_steps(gd, orc, io, key_bytes, runs):
    rng = np.random.default_rng(runs)
    p = Pair(gd, orc, io, key_bytes, 1 << 16)
    # stretches of 0 to 299 dead keys, each behind a live one, in both halves
    # of the key space
    size = rng.permutation(300)
    start = np.concatenate([[0], np.cumsum(size + 2)]).astype(np.uint64)
    keys = np.arange(int(start[-1]), dtype=np.uint64)
    live = np.isin(keys, start)
    keys[len(keys) // 2:] += np.uint64(np.iinfo(p.dt).max // 2)
    keys = keys.astype(p.dt)

    def update(k, gone):
        p.d.apply_mixed(p.up(k), p.up(k ^ p.dt(9)), io.up(gone, np.uint8),
                        count=len(k))
        assert p.o.apply_mixed(k, k ^ p.dt(9), gone.astype(np.uint8)) == 0

    update(keys, np.zeros(len(keys), np.uint8))
    for i in range(1, runs):  # batches of falling size stay runs of their own
        n = len(keys) >> i
        at = rng.choice(len(keys), n, replace=False)
        update(keys[at], (~live[at]).astype(np.uint8))
        q = np.concatenate([keys, [np.iinfo(p.dt).max]]).astype(p.dt)
        assert np.array_equal(successors(p, io, key_bytes, q),
                              p.o.successor(q))
        q = rng.permutation(q)[:-5]
        assert np.array_equal(successors(p, io, key_bytes, q),
                              p.o.successor(q))


@pytest.mark.parametrize("key_bytes", [4, 8])
def test_no_rows(gd, orc, io, key_bytes):
    p = Pair(gd, orc, io, key_bytes, 1000)
    top = np.iinfo(p.dt).max
    for n in (1, 64, 1000):
        q = np.arange(n).astype(p.dt)
        q[-1] = top
        assert np.all(successors(p, io, key_bytes, q) == top)
