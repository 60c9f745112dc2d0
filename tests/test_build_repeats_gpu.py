"""Builds of more than 2^21 32-bit keys, which go by segments where a sample says
that the keys repeat enough, else by radix passes, against the newest update of
each key: keys that come many times shuffled, in copies of the whole input and in
runs, few keys, dense ones, nearly enough repeats, and the keys 0 and 2^32 - 1."""

import numpy as np
import pytest

from test_batch_sort_gpu import keys_of

pytestmark = pytest.mark.gpu


def build_keys(rng, n, kind):
    def some(m):
        return rng.integers(0, 1 << 32, m, dtype=np.uint64).astype(np.uint32)

    if kind == "eight":
        k = rng.choice(some(n // 8), n)
    elif kind == "copies":
        k = np.tile(some(n // 4 + 1), 4)[:n]
    elif kind == "runs of one":
        k = np.repeat(some(n // 5 + 1), 5)[:n]
    elif kind == "near":        # about as many distinct keys as segments take
        k = rng.choice(some(1500000), n)
    elif kind == "few":
        k = rng.choice(some(100), n)
    elif kind == "dense":
        k = rng.integers(0, 300000, n, dtype=np.uint64).astype(np.uint32)
    else:
        k = keys_of(rng, n, kind, 4)
    k[rng.integers(0, n, 50)] = 0
    k[rng.integers(0, n, 50)] = 0xFFFFFFFF
    return k


@pytest.mark.parametrize("kind", ["eight", "copies", "runs of one", "near",
                                  "few", "dense", "full", "hot", "one"])
@pytest.mark.parametrize("n", [(1 << 21) + 1, 2700003])
def test_builds_of_repeated_keys(gd, io, kind, n):
    rng = np.random.default_rng(n)
    k = build_keys(rng, n, kind)
    v = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    # the newest update of each key: the first of the reversed input
    want, first = np.unique(k[::-1], return_index=True)
    want_v = v[::-1][first]
    m = len(want)
    d = gd.GPULSMOpt(max_elements=4 * n, batch_capacity=1 << 20)
    for _ in range(2):
        d.bulk_build(io.up(k), io.up(v), count=n)
        ok, ov = io.empty(m + 1), io.empty(m + 1)
        assert d.dump_sorted(ok, ov, capacity=m + 1) == m
        assert np.array_equal(io.down(ok, m), want)
        assert np.array_equal(io.down(ov, m), want_v)
        q = np.concatenate([rng.choice(want, 30000),
                            rng.integers(0, 1 << 32, 30000, dtype=np.uint64)
                            .astype(np.uint32)])
        at = np.minimum(np.searchsorted(want, q), m - 1)
        out = io.empty(len(q))
        d.lookup(io.up(q), out, count=len(q))
        assert np.array_equal(io.down(out, len(q)),
                              np.where(want[at] == q, want_v[at], 0xFFFFFFFF))
