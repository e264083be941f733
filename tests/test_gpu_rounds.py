"""Launches of all bodies at the sizes where the number of j slices begins to
grow with the i: just above 65536 i, and an odd larger size.  Lists and nearest
neighbours of sampled bodies bit-exact against the oracle, forces within
oracle/parity.py's bar."""
import numpy as np
import pytest

from nbody6ppgpu_amd import gpunb, ics
from oracle import oracle
from oracle.parity import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65536, 65601, 100003])
def test_all_bodies(n):
    c = ics.plummer(n, seed=n, m=ics.kroupa(n, seed=n + 1))
    rs, dtr = ics.neighbour_radii(c, k=20)
    h2 = rs * rs
    gpunb.gpunb_open(n + 10)
    try:
        gpunb.gpunb_send(c.m, c.x, c.v)
        g = gpunb.gpunb_regf(h2, dtr, c.x, c.v, 121, 120, 0, nearest=True)
    finally:
        gpunb.gpunb_close()
    q = np.unique(np.concatenate([np.arange(70), np.arange(0, n, 997),
                                  np.arange(n - 70, n)]))
    o = oracle.regf(c.m, c.x, c.v, h2[q], dtr[q], c.x[q], c.v[q], 121, 120, 0)
    assert_parity(tuple(a[q] for a in g), o, label=f"n={n}",
                  inputs=(c.m, c.x, c.v, c.x[q], c.v[q]))
