"""gpupot_ of all bodies (each 1/r formed once for its pair) against gpupot_
of ranges of them (every pair from its own side) and the oracle, at the sizes
where the block plan changes: 4096 bodies, 128, 512 and 1024 tiles, ragged
last tiles and blocks.  Both paths add the same FP32 tile sums in FP64, in
different orders: at most 1100 tile sums, so 1e-12 relative.  Coincident
bodies, in one tile and in different ones, with and without mass, take no
part in each other's sums."""
import numpy as np
import pytest

from nbody6ppgpu_amd import gpunb, ics
from oracle import oracle
from oracle.parity import FORCE_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4095, 4096, 4097, 8129, 8193, 16385, 32705, 32833, 65537])
@pytest.mark.parametrize("coincident", [False, True])
def test_all_bodies_match_ranges(n, coincident):
    c = ics.plummer(n, seed=n, m=ics.kroupa(n, seed=5))
    m, x = c.m.copy(), c.x.copy()
    if coincident:
        x[1] = x[0]                       # one tile
        x[n - 1] = x[2]                   # first and last tile
        x[n // 2] = x[n // 2 + 64]        # neighbouring tiles
        m[n - 1] = 0.0                    # 0 * inf without the check
        x[70:75] = x[200]                 # several bodies at one point
    whole = gpunb.gpupot(1, n, m, x)
    cut = n // 3
    parts = np.concatenate([gpunb.gpupot(1, cut, m, x), gpunb.gpupot(cut + 1, n - cut, m, x)])
    assert np.all(np.isfinite(whole))
    assert np.max(np.abs(whole - parts) / parts) < 1e-12
    some = np.unique(np.r_[0:4, 70:76, 200, n // 2, n // 2 + 64, n - 2, n - 1])
    for i in some:
        exact = oracle.pot(int(i) + 1, 1, m, x)[0]
        assert abs(whole[i] - exact) < FORCE_TOL * exact
