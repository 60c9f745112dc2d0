"""FliX removes along long chains against the oracle: slices below, at and
beyond the window of staged keys, absent keys between the stored ones, chains
whose nodes all empty (more of them than one return to the ring holds), and an
insert into the nodes that came back."""

import numpy as np
import pytest

from test_flix_gpu import FlixPair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kb,slots", [(4, 16), (4, 64), (8, 32), (8, 64)])
@pytest.mark.parametrize("take", ["all", "tail", "alternate", "absent", "few",
                                  "window"])
def test_removes_along_chains(gd, orc, io, kb, slots, take):
    rng = np.random.default_rng(kb * 100 + slots)
    pair = FlixPair(gd, orc, io, kb, 4, node_slots=slots)
    kt = pair.kt
    heads = (np.arange(1, 601, dtype=np.uint64) << np.uint64(20)).astype(kt)
    pair.build(heads)
    # five stretches each grow a chain of some 90 nodes of 64 slots or more
    big = np.uint64(7) * (np.arange(1, 6001, dtype=np.uint64))
    add = np.concatenate([(big + heads[j]).astype(kt)
                          for j in (3, 4, 5, 400, 598)])
    pair.insert(add, np.arange(len(add), dtype=np.uint32))
    if take == "all":
        gone = add
    elif take == "tail":
        gone = np.concatenate([add[2000:6000], heads[:3]])
    elif take == "alternate":
        gone = add[::2]
    elif take == "absent":    # a node's share is mostly keys it lacks
        gone = np.concatenate([
            add[::5],
            (np.arange(40000, dtype=np.uint64) + heads[4]).astype(kt)])
    elif take == "few":
        gone = add[rng.integers(0, len(add), 40)]
    else:                     # slices of 255, 256, 257 and 513 keys
        gone = np.concatenate([add[6000 * j + 100:6000 * j + 100 + c]
                               for j, c in enumerate((255, 256, 257, 513))])
    pair.remove(rng.permutation(gone))
    pair.check_all(rng, 0, int(heads[-1]) + 50000)
    back = np.concatenate([gone, (add + kt(1))[::3]])
    pair.insert(back, np.arange(len(back), dtype=np.uint32))
    pair.remove(np.sort(add[1::4]), assume_sorted=True)
    pair.check_all(rng, 0, int(heads[-1]) + 50000)
