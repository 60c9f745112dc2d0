"""FliX builds and inserts at the tile edges of the pass that keeps each key's
first occurrence, against the oracle: one key, keys that repeat across tiles,
stretches and distinct keys, 32- and 64-bit keys and values."""

import numpy as np
import pytest

from test_batch_sort_gpu import keys_of
from test_flix_gpu import FlixPair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kb,vb", [(4, 4), (4, 8), (8, 8)])
@pytest.mark.parametrize("kind", ["one", "narrow", "runs", "ascending"])
def test_first_occurrences(gd, orc, io, kb, vb, kind):
    rng = np.random.default_rng(kb + vb)
    for n in (1, 63, 4095, 4096, 4097, 12289, 40960):
        p = FlixPair(gd, orc, io, kb, vb, node_slots=16)
        p.build(keys_of(rng, n, kind, kb) + p.kt(1))
        k = np.concatenate([keys_of(rng, n, kind, kb),
                            keys_of(rng, n // 2 + 1, "full", kb)])
        k = np.maximum(np.minimum(k, np.iinfo(p.kt).max - p.kt(1)), p.kt(1))
        p.insert(k, np.arange(len(k)).astype(p.vt))
        p.check_all(rng, 1, 1 << 24, nq=500)
