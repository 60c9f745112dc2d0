"""Successors over one to many runs (a lane per run), against the oracle: dead
keys in long stretches, keys held by several runs, queries beyond the last key,
the two key widths, and numbers of queries that fill no workgroup."""

import numpy as np
import pytest

from test_batch_sort_gpu import Pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("key_bytes", [4, 8])
@pytest.mark.parametrize("runs", [1, 2, 3, 4, 5, 8, 9])
def test_successors_over_runs(gd, orc, io, key_bytes, runs):
    rng = np.random.default_rng(10 * runs + key_bytes)
    p = Pair(gd, orc, io, key_bytes, 60000)
    top = np.iinfo(p.dt).max
    # batches of falling size stay runs of their own
    for i in range(runs):
        n = 20000 >> i
        k = rng.integers(0, 40000, n, dtype=np.uint64).astype(p.dt)
        k[::7] += p.dt(top // 2)
        if i % 2:   # stretches of dead keys
            k[: n // 2] = np.arange(n // 2).astype(p.dt) + p.dt(1000 * i)
        e = np.zeros(n, np.uint8)
        if i % 2:
            e[: n // 2] = 1
        p.d.apply_mixed(p.up(k), p.up(k ^ p.dt(5)), io.up(e, np.uint8), count=n)
        assert p.o.apply_mixed(k, k ^ p.dt(5), e) == 0
        for m in (1, 63, 257, 5001):
            q = rng.integers(0, 45000, m, dtype=np.uint64).astype(p.dt)
            q[::3] += p.dt(top // 2)
            q[-1] = p.dt(top)
            out = io.empty(m, key_bytes)
            p.d.successor(p.up(q), out, count=m)
            assert np.array_equal(io.down(out, m, p.dt), p.o.successor(q))
