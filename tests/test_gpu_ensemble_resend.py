"""An ensemble sent again with other cluster sizes and other active counts,
and with the same ones: every step's lists bit-exact and forces within
oracle/parity.py's bar against the oracle of each cluster alone."""
import numpy as np
import pytest

from nbody6ppgpu_amd import ensemble, gpunb, ics
from nbody6ppgpu_amd.hiprt import DeviceArray
from oracle import oracle
from oracle.parity import assert_parity

pytestmark = pytest.mark.gpu

CAP = (700, 64, 1, 300)
SIZES = [(700, 64, 1, 300), (65, 63, 0, 129), (65, 63, 0, 129), (640, 1, 1, 64),
         (700, 64, 1, 300)]


def clusters(sizes, seed):
    out = []
    for c, n in enumerate(sizes):
        cl = ics.plummer(max(n, 2), seed=seed + c, m=ics.kroupa(max(n, 2), seed=c) if c % 2 else None)
        rs, dtr = ics.neighbour_radii(cl, k=min(20, max(n - 2, 1)))
        s = slice(0, n)
        out.append((ics.Cluster(cl.m[s], cl.x[s], cl.v[s]), (rs * rs)[s], dtr[s]))
    return out


@pytest.mark.parametrize("persistent", [True, False])
def test_resend(persistent):
    nnbmax = 60
    gpunb.gpunb_ens_open(CAP)
    gpunb.gpunb_ens_persistent(persistent)
    try:
        for step, sizes in enumerate(SIZES):
            cl = clusters(sizes, 50 + step)
            gpunb.gpunb_ens_send([(c.m, c.x, c.v) for c, _, _ in cl])
            b = ensemble.upload(cl, nnbmax)
            ni = [n if step != 2 else (n + 1) // 2 for n in sizes]
            if step == 2:     # half of the bodies active, the same sizes
                cat = lambda f: DeviceArray.from_numpy(np.concatenate(  # noqa: E731
                    [f(c)[:k] for c, k in zip(cl, ni)]))
                b.x, b.v = cat(lambda c: c[0].x), cat(lambda c: c[0].v)
                b.h2, b.dt = cat(lambda c: c[1]), cat(lambda c: c[2])
            ensemble.call(b, ni, nnbmax)
            gpunb.gpunb_sync()
            acc, jrk, pot, nnb, nnid, off, lst = (
                a.numpy() for a in (b.acc, b.jrk, b.pot, b.nnb, b.nnid, b.off, b.lst))
            i0 = 0
            for (c, h2, dt), k in zip(cl, ni):
                s = slice(i0, i0 + k)
                i0 += k
                if k == 0:
                    continue
                o = oracle.regf(c.m, c.x, c.v, h2[:k], dt[:k], c.x[:k], c.v[:k],
                                nnbmax + 1, nnbmax, 0)
                rows = np.zeros((k, nnbmax + 1), np.int32)
                rows[:, 0] = nnb[s]
                for q in range(k):
                    m = nnb[s][q]
                    if m > 0:
                        rows[q, 1:1 + m] = lst[off[s][q]:off[s][q] + m]
                assert_parity((acc[s], jrk[s], pot[s], rows, nnid[s]), o,
                              label=f"step {step} n={c.n}",
                              inputs=(c.m, c.x, c.v, c.x[:k], c.v[:k]))
    finally:
        gpunb.gpunb_ens_persistent(True)
        gpunb.gpunb_ens_close()
