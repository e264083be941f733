"""Sorted order of j and i at the sizes where the sort in runs changes: one
run of 2048 records, one more or less, several, padding records past the
first run, bodies sharing a few sort codes, clusters that begin and end
inside a run.  Lists bit-exact and forces within oracle/parity.py's bar
against the oracle: a record lost or doubled by the sort shows in both."""
import numpy as np
import pytest

from nbody6ppgpu_amd import ensemble, gpunb, ics
from oracle import oracle
from oracle.parity import assert_parity

pytestmark = pytest.mark.gpu


def cluster(n, seed, ties=False):
    c = ics.plummer(n, seed=seed, m=ics.kroupa(n, seed=seed + 1))
    rs, dtr = ics.neighbour_radii(c, k=20)
    if ties:      # one body far out: the rest share a few cells of the box
        c.x[n // 2] = (3e4, 0.0, 0.0)
    return c, rs * rs, dtr


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("n", [1985, 2048, 2049, 2111, 4097, 8200])
def test_one_cluster(n, ties, monkeypatch):
    monkeypatch.setenv("GPUNB_ISORT", "1")     # also below its size
    c, h2, dtr = cluster(n, 30 + n, ties)
    args = (c.m, c.x, c.v, h2, dtr, c.x, c.v, 121, 120, 0)
    gpunb.gpunb_open(n + 10)
    try:
        gpunb.gpunb_send(c.m, c.x, c.v)
        g = gpunb.gpunb_regf(*args[3:], nearest=True)
    finally:
        gpunb.gpunb_close()
    assert_parity(g, oracle.regf(*args), label=f"n={n} ties={ties}",
                  inputs=args[:3] + args[5:7])


@pytest.mark.parametrize("sizes", [(2048, 2048), (2047, 70, 2050, 64, 4100),
                                   (300, 5000, 64)])
def test_ensemble(sizes, monkeypatch):
    monkeypatch.setenv("GPUNB_ISORT", "1")
    nnbmax = 120
    cl = [cluster(n, 60 + k, ties=k == 1) for k, n in enumerate(sizes)]
    gpunb.gpunb_ens_open([n + 70 * (k % 2) for k, n in enumerate(sizes)])
    try:
        gpunb.gpunb_ens_send([(c.m, c.x, c.v) for c, _, _ in cl])
        b = ensemble.upload(cl, nnbmax)
        ensemble.call(b, list(sizes), nnbmax)
        gpunb.gpunb_sync()
        acc, jrk, pot, nnb, nnid, off, lst = (
            a.numpy() for a in (b.acc, b.jrk, b.pot, b.nnb, b.nnid, b.off, b.lst))
    finally:
        gpunb.gpunb_ens_close()
    i0 = 0
    for c, h2, dt in cl:
        k = len(c.m)
        s = slice(i0, i0 + k)
        i0 += k
        o = oracle.regf(c.m, c.x, c.v, h2, dt, c.x, c.v, nnbmax + 1, nnbmax, 0)
        rows = np.zeros((k, nnbmax + 1), np.int32)
        rows[:, 0] = nnb[s]
        for q in range(k):
            m = max(nnb[s][q], 0)
            rows[q, 1:1 + m] = lst[off[s][q]:off[s][q] + m]
        assert_parity((acc[s], jrk[s], pot[s], rows, nnid[s]), o, label=f"{sizes} n={k}",
                      inputs=(c.m, c.x, c.v, c.x, c.v))
