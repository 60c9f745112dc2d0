"""FliX removes whose batch has more keys between two neighbouring nodes' first
keys than a wave's window of staged keys holds (256), with nodes behind them,
against the oracle: dense stretches of mostly absent keys over half-full nodes,
stored keys repeated hundreds of times, and both by turns.  Long chains in
neighbouring buckets go to neighbouring waves of one workgroup."""

import numpy as np
import pytest

from test_flix_gpu import FlixPair

pytestmark = pytest.mark.gpu

WINDOW = 256
STRIDE = 80


def shares(nodes_first, batch):
    """Keys of the batch from each node's first key up to the next one's."""
    return np.diff(np.searchsorted(batch, nodes_first))


@pytest.mark.parametrize("kb,slots", [(4, 16), (8, 16), (4, 32), (8, 32),
                                      (4, 40), (4, 64), (8, 64)])
@pytest.mark.parametrize("kind", ["dense", "first", "every", "turns"])
@pytest.mark.parametrize("presorted", [False, True])
def test_shares_beyond_the_window(gd, orc, io, kb, slots, kind, presorted):
    rng = np.random.default_rng(kb * 100 + slots)
    pair = FlixPair(gd, orc, io, kb, 4, node_slots=slots,
                    rebuild_chain_nodes=0)
    kt = pair.kt
    heads = (np.arange(1, 601, dtype=np.uint64) << np.uint64(20)).astype(kt)
    pair.build(heads)
    # a long chain in each of the neighbouring buckets (a build fills them
    # with slots / 2 heads); chains that an insert grows have half-full nodes
    grown = heads[::slots // 2]
    per = 20 * (slots // 2)  # some 20 nodes
    off = np.arange(1, per + 1, dtype=np.uint64) * np.uint64(STRIDE)
    add = np.concatenate([(off + h).astype(kt) for h in grown])
    pair.insert(add, np.arange(len(add), dtype=np.uint32))
    one = off[:per // 2 + 7]                 # up to the middle of a chain
    if kind == "dense":
        rel = np.arange(int(one[-1]) + 1, dtype=np.uint64)
    elif kind == "first":                    # one key, then all the others
        rel = np.concatenate([np.repeat(off[:1], 300), one])
    elif kind == "every":
        rel = np.repeat(off, rng.integers(1, 150, len(off)))
    else:                                    # a dense stretch, then a gap
        rel = np.arange(int(off[-1]), dtype=np.uint64)
        rel = rel[(rel // np.uint64(5 * STRIDE * slots)) % np.uint64(2) == 0]
    gone = np.concatenate([(rel + h).astype(kt) for h in grown])
    firsts = off[::slots // 2] + grown[0].astype(np.uint64)
    assert shares(firsts, np.sort(gone)).max() > WINDOW
    pair.remove(np.sort(gone) if presorted else rng.permutation(gone),
                assume_sorted=presorted)
    pair.check_all(rng, 0, int(heads[-1]) + 50000)
    # the nodes that came back serve an insert, and empty again
    pair.insert(add, np.arange(len(add), dtype=np.uint32)[::-1].copy())
    pair.remove(np.sort(np.repeat(add, 9)), assume_sorted=True)
    pair.check_all(rng, 0, int(heads[-1]) + 50000)
