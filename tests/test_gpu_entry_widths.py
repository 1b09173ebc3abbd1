"""Entries at every remainder of the widths in which a slice's terms are loaded (1, 2, 4,
8, 16, 32): ranks that differ along the train, bit for bit against the oracle's chain."""
import numpy as np
import pytest

import oracle_lib as O
import paratt_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", list(range(1, 35)) + [40, 41, 48, 49, 63, 64, 65, 96, 97])
def test_entry(r):
    n, ranks = [5, 4, 6, 3, 7], [1, max(1, r - 1), r, r + 1, max(1, r // 2), 1]
    x = O.gauss_tt(n, ranks, r, 0.5)
    dx = P.DevTT.from_host(x)
    rng = np.random.default_rng(r)
    for _ in range(4):
        idx = [int(rng.integers(0, m)) for m in n]
        assert P.entry(dx, idx) == O.entry(x, idx)
