"""The merges of the sort in runs (csrc/sort_merge.h) on the CPU, against a
stable sort: one cluster at one run of 1024 records and at the 32 runs of the
last merge, clusters of an ensemble at the 15360 records that it takes whole,
one less and one more of each, ties and padding records among them."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "nbody6ppgpu_amd", "csrc")
PAD = 0xffffffff


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("sort") / "sort_merge_cpu.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-w", "-shared", "-fPIC",
                           "-I/opt/rocm/include", "-I" + CSRC,
                           os.path.join(HERE, "sort_merge_cpu.cpp"), "-o", so])
    return ctypes.CDLL(so)


def codes(n, distinct, pad, rng):
    """n codes of at most `distinct` values, some of heavy bodies, the last
    `pad` those of padding records."""
    k = rng.integers(0, distinct, n, dtype=np.uint32)
    k |= (rng.random(n) < 0.02).astype(np.uint32) << np.uint32(30)
    if pad:
        k[max(n - pad, 0):] = PAD
    return k


def ip(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 2048, 2049, 16385,
                               32704, 32767, 32768, 32769, 32832, 70001])
def test_one_cluster(lib, n):
    rng = np.random.default_rng(n)
    assert lib.merges_before_last(n, n, 1) == (n > 32768)
    for distinct in (1, 3, 1000, 1 << 30):
        for pad in (0, 37):
            for in_order in (False, True):
                k = codes(n, distinct, pad, rng)
                if in_order:
                    k.sort()
                order = np.empty(n, np.int32)
                assert lib.sort_one(n, k.ctypes.data_as(ctypes.c_void_p),
                                    ip(order)) == 0
                assert np.array_equal(order, np.argsort(k, kind="stable"))


def test_one_cluster_with_two_merges_before_the_last(lib):
    n = 32 * 32768 + 1
    assert lib.merges_before_last(n, n, 1) == 2
    k = codes(n, 1 << 30, 63, np.random.default_rng(1))
    order = np.empty(n, np.int32)
    assert lib.sort_one(n, k.ctypes.data_as(ctypes.c_void_p), ip(order)) == 0
    assert np.array_equal(order, np.argsort(k, kind="stable"))


@pytest.mark.parametrize("sizes", [
    (15360, 15360), (15361, 15361), (1, 15360, 64), (1023, 15360, 15360, 5),
    (1, 15361, 64), (1023, 15361, 15359, 5), (64, 0, 0, 40000, 1, 128, 0),
    (15360,) * 4, (100,) * 70, (1024,) * 33, (0, 3, 0)])
def test_clusters(lib, sizes):
    rng = np.random.default_rng(sum(sizes) + len(sizes))
    n, n_max = sum(sizes), max(sizes)
    assert lib.merges_before_last(n, n_max, 0) == (n_max > 15360)
    c0 = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    for distinct in (1, 5, 1 << 30):
        for pad in (0, 70):
            k = np.concatenate([
                np.uint64(c << 32) | codes(s, distinct, pad if c % 2 else 0, rng).astype(np.uint64)
                for c, s in enumerate(sizes)])
            order = np.empty(n, np.int32)
            assert lib.sort_clusters(n, k.ctypes.data_as(ctypes.c_void_p), n_max,
                                     ip(c0), ip(order)) == 0
            assert np.array_equal(order, np.argsort(k, kind="stable"))
