"""Batches that one workgroup admits, against the oracle: sizes around the
items per thread and the capacity, keys of which few digits vary, repeated
keys, and erases (alone and mixed with inserts)."""

import numpy as np
import pytest

from test_batch_sort_gpu import KINDS, Pair, keys_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("key_bytes", [4, 8])
def test_small_batches(gd, orc, io, kind, key_bytes):
    rng = np.random.default_rng(key_bytes)
    p = Pair(gd, orc, io, key_bytes, 1 << 16)
    sizes = [1, 2, 63, 64, 65, 511, 512, 513, 700, 1024, 1025, 2047, 2048]
    if key_bytes == 4:
        sizes += [2049, 3585, 4095, 4096]
    for i, n in enumerate(sizes):
        k = keys_of(rng, n, kind, key_bytes)
        v = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(p.dt)
        e = (rng.random(n) < 0.25).astype(np.uint8)
        if i % 4 == 1:
            p.d.erase(p.up(k[::2]), count=len(k[::2]))
            assert p.o.erase(k[::2]) == 0
        if i % 2:
            p.d.apply_mixed(p.up(k), p.up(v), io.up(e, np.uint8), count=n)
            assert p.o.apply_mixed(k, v, e) == 0
        else:
            p.d.insert(p.up(k), p.up(v), count=n)
            assert p.o.insert(k, v) == 0
        p.check(rng)
