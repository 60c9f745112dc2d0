"""Long ranges at the edge of the launches whose groups of queries get a team of
workgroups (1024 queries) against prefix sums of the oracle's contents, by turns
on one handle, as the teams' sums start from zero in each call."""

import numpy as np
import pytest

from test_long_ranges_gpu import Filled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("key_bytes", [4, 8])
def test_edge_of_the_teams(gd, orc, io, key_bytes):
    f = Filled(gd, orc, io, key_bytes, [140000, 5000], 0.1, False, 6)
    rng = np.random.default_rng(8)
    for n in (1023, 1024, 1025, 1, 1024, 1021, 2048, 1024):
        i = rng.integers(0, len(f.keys) - 2500, n)
        f.check(f.keys[i], f.keys[i + rng.integers(2, 2500, n)])
