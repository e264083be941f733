"""Sorted order of j and i on both sides of the sizes where the sort's launches
change: one run of 1024 records, the 32 runs (32768 records) that the last merge
of one cluster takes, the 15360 records of an ensemble's cluster above which
another merge comes before the last, clusters that begin inside a run.  Lists
bit-exact and forces within oracle/parity.py's bar against the oracle: a record
lost or doubled by the sort shows in both."""
import numpy as np
import pytest

from nbody6ppgpu_amd import ensemble, gpunb, ics
from oracle import oracle
from oracle.parity import assert_parity

pytestmark = pytest.mark.gpu

NNBMAX = 120


def cluster(n, seed):
    c = ics.plummer(n, seed=seed, m=ics.kroupa(n, seed=seed + 1))
    rs, dtr = ics.neighbour_radii(c, k=20)
    return c, rs * rs, dtr


@pytest.mark.parametrize("n", [960, 1023, 1024, 1025, 32768, 32769])
def test_one_cluster(n, monkeypatch):
    monkeypatch.setenv("GPUNB_ISORT", "1")     # also below its size
    c, h2, dtr = cluster(n, 30 + n)
    args = (c.m, c.x, c.v, h2, dtr, c.x, c.v, NNBMAX + 1, NNBMAX, 0)
    gpunb.gpunb_open(n + 10)
    try:
        gpunb.gpunb_send(c.m, c.x, c.v)
        g = gpunb.gpunb_regf(*args[3:], nearest=True)
    finally:
        gpunb.gpunb_close()
    assert_parity(g, oracle.regf(*args), label=f"n={n}")


@pytest.mark.parametrize("sizes", [(15360, 300), (15361, 300), (100, 15360, 64),
                                   (100, 15361, 64)])
def test_ensemble(sizes, monkeypatch):
    monkeypatch.setenv("GPUNB_ISORT", "1")
    cl = [cluster(n, 60 + k) for k, n in enumerate(sizes)]
    gpunb.gpunb_ens_open(list(sizes))
    try:
        gpunb.gpunb_ens_send([(c.m, c.x, c.v) for c, _, _ in cl])
        b = ensemble.upload(cl, NNBMAX)
        ensemble.call(b, list(sizes), NNBMAX)
        gpunb.gpunb_sync()
        acc, jrk, pot, nnb, nnid, off, lst = (
            a.numpy() for a in (b.acc, b.jrk, b.pot, b.nnb, b.nnid, b.off, b.lst))
    finally:
        gpunb.gpunb_ens_close()
    i0 = 0
    for c, h2, dt in cl:
        k = c.n
        s = slice(i0, i0 + k)
        i0 += k
        o = oracle.regf(c.m, c.x, c.v, h2, dt, c.x, c.v, NNBMAX + 1, NNBMAX, 0)
        rows = np.zeros((k, NNBMAX + 1), np.int32)
        rows[:, 0] = nnb[s]
        for q in range(k):
            m = max(nnb[s][q], 0)
            rows[q, 1:1 + m] = lst[off[s][q]:off[s][q] + m]
        assert_parity((acc[s], jrk[s], pot[s], rows, nnid[s]), o, label=f"{sizes} n={k}")
