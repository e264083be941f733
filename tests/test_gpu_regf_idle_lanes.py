"""Mass-weighted lists of calls whose last wavefront has idle lanes, with a
massive body at the origin, where an idle lane's position is: the mass-weighted
screen flags the pair of the two.  The call, the next one with more i on the
same engine, and the next cluster of an ensemble have to list what the FP64
oracle lists, and no more: lists and nearest neighbours bit-exact, forces within
oracle/parity.py's bar."""
import numpy as np
import pytest

from nbody6ppgpu_amd import ensemble, gpunb, ics
from oracle import oracle
from oracle.parity import assert_parity

pytestmark = pytest.mark.gpu

NNBMAX = 150


def cluster(n, seed):
    """Kroupa masses; body n // 2 is a hundred mean masses at rest at the
    origin."""
    c = ics.plummer(n, seed=seed, m=ics.kroupa(n, seed=seed + 1))
    rs, dtr = ics.neighbour_radii(c, k=12)
    c.m[n // 2] = 100.0 * np.mean(c.m)
    c.x[n // 2] = 0.0
    c.v[n // 2] = 0.0
    return c, rs * rs / np.mean(c.m), dtr


@pytest.mark.parametrize("prec", [65, 32])
@pytest.mark.parametrize("blocks", [(1, 64, 65), (65, 130, 700), (700, 63, 128)])
def test_next_call_finds_no_entries(blocks, prec, monkeypatch):
    monkeypatch.setenv("GPUNB_ISORT", "1" if prec == 32 else "0")
    n = 700
    c, h2, dtr = cluster(n, 91)
    order = np.random.default_rng(92).permutation(n)
    gpunb.gpunb_set_precision(prec)
    gpunb.gpunb_open(n + 10)
    try:
        gpunb.gpunb_send(c.m, c.x, c.v)
        for ni in blocks:
            i = order[:ni]
            args = (c.m, c.x, c.v, h2[i], dtr[i], c.x[i], c.v[i],
                    NNBMAX + 1, NNBMAX, 1)
            g = gpunb.gpunb_regf(*args[3:], nearest=True)
            assert_parity(g, oracle.regf(*args), label=f"ni={ni} of {blocks} {prec}",
                          inputs=args[:3] + args[5:7])
    finally:
        gpunb.gpunb_close()
        gpunb.gpunb_set_precision(0)


@pytest.mark.parametrize("prec", [65, 32])
@pytest.mark.parametrize("persistent", [True, False])
def test_next_cluster_finds_no_entries(persistent, prec):
    sizes = (300, 129, 65, 700, 1)
    cl = [cluster(n, 93 + k) for k, n in enumerate(sizes)]
    gpunb.gpunb_set_precision(prec)
    gpunb.gpunb_ens_open([n + 10 for n in sizes])
    gpunb.gpunb_ens_persistent(persistent)
    try:
        gpunb.gpunb_ens_send([(c.m, c.x, c.v) for c, _, _ in cl])
        b = ensemble.upload(cl, NNBMAX)
        ni = np.array(sizes, dtype=np.int32)
        for _ in range(2):     # the second call finds the counts reset
            rc = gpunb.load().gpunb_ens_regf_dev(
                len(ni), ni.ctypes.data_as(gpunb._ip), b.h2.ptr, b.dt.ptr,
                b.x.ptr, b.v.ptr, b.acc.ptr, b.jrk.ptr, b.pot.ptr, NNBMAX, 1,
                b.nnb.ptr, b.nnid.ptr, b.lst.ptr, b.off.ptr, b.total.ptr, b.cap)
            if rc != 0:
                gpunb._check()
        gpunb.gpunb_sync()
        acc, jrk, pot, nnb, nnid, off, lst = (
            a.numpy() for a in (b.acc, b.jrk, b.pot, b.nnb, b.nnid, b.off, b.lst))
    finally:
        gpunb.gpunb_ens_persistent(True)
        gpunb.gpunb_ens_close()
        gpunb.gpunb_set_precision(0)
    i0 = 0
    for c, h2, dt in cl:
        k = c.n
        s = slice(i0, i0 + k)
        i0 += k
        o = oracle.regf(c.m, c.x, c.v, h2, dt, c.x, c.v, NNBMAX + 1, NNBMAX, 1)
        rows = np.zeros((k, NNBMAX + 1), np.int32)
        rows[:, 0] = nnb[s]
        for q in range(k):
            m = max(nnb[s][q], 0)
            rows[q, 1:1 + m] = lst[off[s][q]:off[s][q] + m]
        assert_parity((acc[s], jrk[s], pot[s], rows, nnid[s]), o,
                      label=f"n={k} persistent={persistent} {prec}",
                      inputs=(c.m, c.x, c.v, c.x, c.v))
