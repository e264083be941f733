"""Batches of the irregular force in the order of the calls, where they take
different ways: up to eight are blocks of their own, large ones (256 KiB and
more) uploaded, small ones read where they are, and the others are merged.  The
last value of a body wins, whichever way it came: the forces of 40 bodies
against the oracle, and the same bits as one batch of the final values."""
import numpy as np
import pytest

from nbody6ppgpu_amd import gpunb
from oracle import oracle
from test_gpu_irr import check, knn_lists, scales, state

pytestmark = pytest.mark.gpu

N = 3000          # a batch of all: 348 KB of records, 312 KB of rows


def test_batches_apply_in_order():
    m, x, v, f, fd, t0 = state(N, 51)
    lists = knn_lists(x, 25)
    one = [np.asarray(l, np.int32) + 1 for l in lists]
    idx = np.arange(N)
    act = idx[::75]

    def put(s, dx=0.0):
        gpunb.irr_set_jp(s + 1, x[s] + dx, v[s], f[s], fd[s], m[s], t0[s])

    def rows(s, shift=0):
        gpunb.irr_set_lists(s + 1, [one[(i + shift) % N] for i in s])

    def small(dx=0.0, shift=0):
        for s in np.array_split(idx, 30):
            put(s, dx)
            rows(s, shift)

    def large(dx=0.0, shift=0):
        put(idx, dx)
        rows(idx, shift)

    want = oracle.irr(0.001, act, t0, x, v, f, fd, m, lists)
    sc = scales(0.001, act, t0, x, v, f, fd, m, lists)
    gpunb.irr_open(N, 40)
    try:
        large()
        first = gpunb.irr_firr(0.001, act + 1)
        check(first, want, sc)
        for stale in ([large] * 11, [small] * 2, [small, large], [large, small],
                      [large] * 3 + [small] + [large] * 2):
            for last in (large, small):
                for k, way in enumerate(stale):
                    way(1.0 + k, 1 + k)
                last()
                got = gpunb.irr_firr(0.001, act + 1)
                assert all(np.array_equal(a, b) for a, b in zip(first, got))
    finally:
        gpunb.irr_close()
