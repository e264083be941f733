"""Batched staging of the irregular force (gpunb_irr_set_jp / _set_lists):
the same bits as per-body batches (the per-particle staging) at the sizes
where the path changes (64 bodies per block, 256 KiB per upload, 2 MiB per
split copy, 2048 bodies with results written directly, 32768 with results in
parts), in the order of the calls, and refused without a trace."""
import numpy as np
import pytest

from nbody6ppgpu_amd import gpunb
from oracle import oracle
from test_gpu_irr import check, knn_lists, scales, state

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(p, q) for p, q in zip(a, b))


@pytest.mark.parametrize("n", [63, 64, 65, 2047, 2049, 2400, 20001, 33000])
def test_blocks_match_single_staging(n):
    m, x, v, f, fd, t0 = state(n, 30 + n)
    lists = knn_lists(x, min(33, n - 2))
    one = [np.asarray(l, np.int32) + 1 for l in lists]
    addr = np.random.default_rng(n).permutation(n) + 1
    k = addr - 1
    got = []
    for step in (n, 50):           # all at once; batches too small for blocks
        gpunb.irr_open(n, 40)
        try:
            for q in range(0, n, step):
                s = k[q:q + step]
                gpunb.irr_set_jp(s + 1, x[s], v[s], f[s], fd[s], m[s], t0[s])
                gpunb.irr_set_lists(s + 1, [one[i] for i in s])
            got.append(gpunb.irr_firr(0.003, addr))
        finally:
            gpunb.irr_close()
    assert same(*got)
    some = k[:200]
    want = oracle.irr(0.003, some, t0, x, v, f, fd, m, lists)
    check([g[:200] for g in got[0]], want,
          scales(0.003, some, t0, x, v, f, fd, m, lists))


def test_calls_apply_in_order():
    """Blocks, repeated blocks (more than are kept), a body listed twice in a
    batch, single calls before and after a batch: the last value wins."""
    n = 500
    m, x, v, f, fd, t0 = state(n, 41)
    lists = knn_lists(x, 20)
    one = [np.asarray(l, np.int32) + 1 for l in lists]
    idx = np.arange(n)
    put = lambda s, dx=0.0: gpunb.irr_set_jp(  # noqa: E731
        s + 1, x[s] + dx, v[s], f[s], fd[s], m[s], t0[s])
    lst = lambda s, w: gpunb.irr_set_lists(s + 1, w)  # noqa: E731
    want = oracle.irr(0.001, idx, t0, x, v, f, fd, m, lists)
    sc = scales(0.001, idx, t0, x, v, f, fd, m, lists)
    gpunb.irr_open(n, 40)
    try:
        for r in range(11):
            put(idx, 1.0 + r)
            lst(idx, [one[(i + r + 1) % n] for i in idx])
        put(idx)
        lst(idx, one)
        check(gpunb.irr_firr(0.001, idx + 1), want, sc)
        put(idx, 3.0)                              # block, then singles
        for i in idx:
            put(np.array([i]))
        check(gpunb.irr_firr(0.001, idx + 1), want, sc)
        put(np.array([7]), 5.0)                    # a single, then a block
        lst(np.array([9]), [one[3]])
        put(idx)
        lst(idx, one)
        check(gpunb.irr_firr(0.001, idx + 1), want, sc)
        twice = np.r_[idx, idx[:80]]               # listed twice in one batch
        gpunb.irr_set_jp(twice + 1, np.r_[x + 2.0, x[:80]], np.r_[v, v[:80]],
                         np.r_[f, f[:80]], np.r_[fd, fd[:80]],
                         np.r_[m, m[:80]], np.r_[t0, t0[:80]])
        put(idx[80:])
        lst(twice, [one[(i + 1) % n] for i in idx] + one[:80])
        lst(idx[80:], one[80:])
        check(gpunb.irr_firr(0.001, idx + 1), want, sc)
    finally:
        gpunb.irr_close()


def test_refused_batches_leave_nothing():
    n = 300
    m, x, v, f, fd, t0 = state(n, 42)
    lists = knn_lists(x, 20)
    one = [np.asarray(l, np.int32) + 1 for l in lists]
    idx = np.arange(n)
    gpunb.irr_open(n, 40)
    try:
        gpunb.irr_set_jp(idx + 1, x, v, f, fd, m, t0)
        gpunb.irr_set_lists(idx + 1, one)
        first = gpunb.irr_firr(0.001, idx + 1)
        bad = idx + 1
        for wrong in (0, n + 1):
            bad[-1] = wrong
            with pytest.raises(gpunb.GpunbError):
                gpunb.irr_set_jp(bad, x + 1.0, v, f, fd, m, t0)
            with pytest.raises(gpunb.GpunbError):
                gpunb.irr_set_lists(bad, one)
            with pytest.raises(gpunb.GpunbError):
                gpunb.irr_set_lists(idx + 1, one[:-1] + [np.array([wrong], np.int32)])
        with pytest.raises(gpunb.GpunbError):
            gpunb.irr_set_lists(idx + 1, one[:-1] + [np.ones(41, np.int32)])
        assert same(first, gpunb.irr_firr(0.001, idx + 1))
    finally:
        gpunb.irr_close()
