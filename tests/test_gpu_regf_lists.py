"""Neighbour lists of the regular force at the sizes where the list paths
change: entries kept in LDS and appended in batches (14 rows per wavefront),
lists of one entry per lane (up to 64) and longer ones sorted in chunks,
lists at and past nnbmax, and calls whose j slices are cut finer than a tile.
Lists and nearest neighbours bit-exact against the FP64 oracle, forces within
oracle/parity.py's bar."""
import numpy as np
import pytest

from nbody6ppgpu_amd import gpunb, ics
from oracle import oracle
from oracle.parity import assert_parity

pytestmark = pytest.mark.gpu

LENGTHS = (1, 2, 3, 13, 14, 15, 28, 29, 63, 64, 65, 127, 128, 129, 193, 300, 301)


def lengths_h2(x, xi, lengths):
    """h2 of each i between its k-th and (k+1)-th nearest body, k cycling
    through lengths (the body itself counts)."""
    d2 = np.sum((xi[:, None, :] - x[None, :, :]) ** 2, axis=2)
    d2.sort(axis=1)
    k = np.array([lengths[q % len(lengths)] for q in range(len(xi))])
    k = np.minimum(k, len(x))
    q = np.arange(len(xi))
    return np.where(k < len(x), 0.5 * (d2[q, k - 1] + d2[q, np.minimum(k, len(x) - 1)]),
                    d2[q, -1] * 1.01 + 1e-9)


@pytest.mark.parametrize("prec", [65, 32])
@pytest.mark.parametrize("m_flag", [0, 1])
@pytest.mark.parametrize("nj,ni,nnbmax", [(60, 60, 64), (64, 20, 63), (1000, 20, 300),
                                          (1000, 65, 301), (4097, 130, 300),
                                          (70000, 17, 300)])
def test_list_lengths(nj, ni, nnbmax, m_flag, prec):
    c = ics.plummer(nj, seed=7 + nj, m=ics.kroupa(nj, seed=8) if m_flag else None)
    xi, vi = c.x[:ni].copy(), c.v[:ni].copy()
    h2 = lengths_h2(c.x, xi, LENGTHS)
    if m_flag:
        h2 = h2 / np.mean(c.m)
    args = (c.m, c.x, c.v, h2, np.zeros(ni), xi, vi, nnbmax + 1, nnbmax, m_flag)
    gpunb.gpunb_set_precision(prec)
    gpunb.gpunb_open(nj + 10)
    try:
        gpunb.gpunb_send(c.m, c.x, c.v)
        for _ in range(2):     # the second call finds the counts reset
            g = gpunb.gpunb_regf(*args[3:], nearest=True)
    finally:
        gpunb.gpunb_close()
        gpunb.gpunb_set_precision(0)
    assert_parity(g, oracle.regf(*args), label=f"nj={nj} ni={ni} m_flag={m_flag} {prec}",
                  inputs=args[:3] + args[5:7])
