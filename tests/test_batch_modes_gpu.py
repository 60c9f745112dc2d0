"""Inserts, mixed updates and erases of batches around the sizes where the
admission of 32-bit keys changes (one workgroup up to 8192 keys, segments from
there on), and of 64-bit ones, each in every mode, against the oracle."""

import numpy as np
import pytest

from test_batch_sort_gpu import KINDS, Pair, keys_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("key_bytes,n", [
    (4, 4097), (4, 8191), (4, 8192), (4, 8193), (4, 12289), (4, 16383),
    (4, 16384), (4, 16385), (8, 6145), (8, 30011)])
def test_every_mode(gd, orc, io, kind, key_bytes, n):
    rng = np.random.default_rng(n + key_bytes)
    k = keys_of(rng, n, kind, key_bytes)
    v = rng.integers(0, 1 << 63, n, dtype=np.uint64).astype(k.dtype)
    e = (rng.random(n) < 0.25).astype(np.uint8)
    p = Pair(gd, orc, io, key_bytes, n)
    p.d.apply_mixed(p.up(k), p.up(v), io.up(e, np.uint8), count=n)
    assert p.o.apply_mixed(k, v, e) == 0
    p.check(rng)
    gone = keys_of(rng, n, kind, key_bytes)
    gone[: n // 2] = rng.permutation(k)[: n // 2]
    p.d.erase(p.up(gone), count=n)
    assert p.o.erase(gone) == 0
    p.check(rng)
    k = rng.permutation(k)
    p.d.insert(p.up(k), p.up(v), count=n)
    assert p.o.insert(k, v) == 0
    p.check(rng)
