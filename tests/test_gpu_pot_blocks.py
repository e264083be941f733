"""gpupot_ of all bodies where a block of bodies is walked in several groups of
tiles (more than 131072 bodies): whole and ragged last blocks and groups, and a
last block of one tile, against gpupot_ of ranges of the bodies and the oracle.
Both add the same FP32 tile sums in FP64, in different orders: at most 4300 of
them, each rounding 1.1e-16 of the sum, so 1e-12 relative."""
import numpy as np
import pytest

from nbody6ppgpu_amd import gpunb, ics
from oracle import oracle
from oracle.parity import FORCE_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [131072, 131073, 150001, 163841, 270001])
def test_all_bodies_match_ranges(n):
    c = ics.plummer(n, seed=n, m=ics.kroupa(n, seed=6))
    m, x = c.m.copy(), c.x.copy()
    x[n - 1] = x[2]                   # coincident, first and last block
    x[n // 2] = x[n // 2 + 640]
    whole = gpunb.gpupot(1, n, m, x)
    cut = n // 3
    parts = np.concatenate([gpunb.gpupot(1, cut, m, x),
                            gpunb.gpupot(cut + 1, n - cut, m, x)])
    assert np.max(np.abs(whole - parts) / parts) < 1e-12
    for i in (0, 2, n // 2, n // 2 + 640, n - 2, n - 1):
        exact = oracle.pot(i + 1, 1, m, x)[0]
        assert abs(whole[i] - exact) < FORCE_TOL * exact
