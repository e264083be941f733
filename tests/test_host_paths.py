"""Host paths of libgpunb.so that need no kernel to run, on the CPU:
hip_host_stub.cpp takes the place of the HIP runtime (in a process of its own),
fails the allocations and copies that a test names and records what the library
launched, held and destroyed."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PREAMBLE = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_most_device.argtypes = [ctypes.c_size_t]
stub.stub_most_pinned.argtypes = [ctypes.c_size_t]
stub.stub_held_device.restype = ctypes.c_size_t
import numpy as np
from nbody6ppgpu_amd import gpunb
gpunb.load()

def refused(fn, *a):
    try:
        fn(*a)
    except gpunb.GpunbError:
        return True
    return False
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_host_stub.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-w", "-shared", "-fPIC",
                           "-I/opt/rocm/include",
                           os.path.join(HERE, "hip_host_stub.cpp"), "-o", so])
    return so


def run(stub, body):
    env = dict(os.environ, PYTHONPATH=ROOT, GPUNB_QUIET="1")
    r = subprocess.run([sys.executable, "-c", PREAMBLE + textwrap.dedent(body), stub],
                       env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}{r.stderr}"


def test_graph_is_not_destroyed_while_it_runs(stub):
    """Other pointers, and another table of slices, after a launch that
    nothing has waited for."""
    run(stub, """
        from nbody6ppgpu_amd import ensemble, ics
        from nbody6ppgpu_amd import hiprt

        class Host:             # device arrays are host memory here
            def __init__(self, shape, dtype):
                self.a = np.zeros(shape, dtype)
                self.ptr = self.a.ctypes.data
            from_numpy = staticmethod(lambda a: Host(a.shape, a.dtype))
        ensemble.DeviceArray = Host

        cl = []
        for n in (100, 70):
            c = ics.plummer(n, seed=n)
            cl.append((c, np.ones(n), np.zeros(n)))
        gpunb.gpunb_ens_open([100, 70])
        gpunb.gpunb_ens_graph(True)
        gpunb.gpunb_ens_send([(c.m, c.x, c.v) for c, _, _ in cl])
        b = ensemble.upload(cl, 20)
        for _ in range(2):
            ensemble.call(b, [100, 70], 20)
        other = ensemble.upload(cl, 20)
        ensemble.call(other, [100, 70], 20)
        gpunb.gpunb_ens_set_bucket_tiles([1] * 24)
        ensemble.call(other, [100, 70], 20)
        gpunb.gpunb_ens_close()
        assert stub.stub_graph_faults() == 0, stub.stub_graph_faults()
    """)


IRR = """
    n = 6000
    gpunb.irr_open(n, 40)
    idx = np.arange(n)
    x = np.zeros((n, 3))
    m = np.zeros(n)
    rows = [np.array([1 + (i + 1) % n], np.int32) for i in range(n)]

    def jp(s):
        gpunb.irr_set_jp(s + 1, x[s], x[s], x[s], x[s], m[s], m[s])

    def lists(s):
        gpunb.irr_set_lists(s + 1, [rows[i] for i in s])
"""


def test_irr_refused_upload_stages_nothing(stub):
    """Records and rows of per-particle calls whose upload finds no memory, or
    fails: an error, and the next call sends them."""
    run(stub, IRR + """
    one = [np.array([i]) for i in range(3000)]
    full = [np.arange(1, 31, dtype=np.int32)] * n
    rows = full                                   # rows of 372 KB in all
    for fault in ("memory", "copy"):
        for s in one:
            jp(s)
            lists(s)
        if fault == "memory":
            stub.stub_most_device(200 << 10)
        else:
            stub.stub_fail_uploads(1)
        assert refused(gpunb.irr_firr, 0.0, idx[:100] + 1)
        stub.stub_most_device(1 << 40)
        if fault == "copy":
            for s in one:         # newer rows of the same bodies
                lists(s)
            stub.stub_fail_uploads(1)
            assert refused(gpunb.irr_firr, 0.0, idx[:100] + 1)
        gpunb.irr_firr(0.0, idx[:100] + 1)
        assert stub.stub_null_args() == 0
        assert stub.stub_launches(b"k_irr_stage") > 0
    """)


def test_irr_buffer_that_did_not_grow_is_not_used(stub):
    """A batch that needs larger buffers than there is memory for is refused,
    and smaller ones after it are staged in buffers of their own."""
    run(stub, IRR + """
    for limit, most in ((stub.stub_most_device, 5000), (stub.stub_most_pinned, 6000)):
        jp(idx[:3000])
        gpunb.irr_firr(0.0, idx[:10] + 1)
        limit(116 * most - 1)
        assert refused(jp, idx[:most])
        limit(1 << 40)
        jp(idx[:3000])
        gpunb.irr_firr(0.0, idx[:10] + 1)
        assert stub.stub_null_args() == 0
    gpunb.irr_close()
    """)


def test_irr_split_copy_without_memory_for_threads(stub):
    """A batch whose copy is split over threads, with every allocation made
    inside the call failing in its turn (the first is the entry point's own,
    before it), without buffers and with those of an earlier call: staged or
    refused, the process going on."""
    run(stub, IRR.replace("n = 6000", "n = 20000") + """
    assert 116 * n >= 2 << 20
    for again in range(2):
        for k in range(1, 10):
            stub.stub_fail_new(k)
            done = not refused(jp, idx)
            stub.stub_fail_new(-1)
            gpunb.irr_firr(0.0, idx[:10] + 1)
            assert stub.stub_null_args() == 0
            assert done or not again
        assert done
    gpunb.irr_close()
    """)


def test_potential_without_memory_for_its_partials(stub):
    """All bodies, with too little device memory for the partials of the
    kernel that forms each 1/r once: the other kernel, not an error; and
    gpunb_close_ gives the partials back."""
    run(stub, """
        n = 40000
        m, x = np.ones(n), np.zeros((n, 3))
        gpunb.gpunb_open(100)
        held = stub.stub_held_device()
        stub.stub_most_device(30 << 20)
        gpunb.gpupot(1, n, m, x)
        assert stub.stub_launches(b"k_pot_sym") == 0
        assert stub.stub_launches(b"k_pot_pass1") == 1
        stub.stub_most_device(1 << 40)
        gpunb.gpupot(1, n, m, x)
        assert stub.stub_launches(b"k_pot_sym") == 1
        assert stub.stub_held_device() > held + (90 << 20)
        gpunb.gpunb_close()
        gpunb.gpunb_open(100)
        assert stub.stub_held_device() < held + (4 << 20)
    """)


def test_irr_batches_allocate_once(stub):
    """The same batches again and again, more of them than are blocks of their
    own, and single calls: no allocation after the first call."""
    run(stub, IRR + """
    def call():
        for s in np.split(idx[:1000], 10):
            jp(s)
            lists(s)
        jp(idx)
        lists(idx)
        jp(idx[:1])
        gpunb.irr_firr(0.0, idx[:1000] + 1)

    for _ in range(2):
        call()
    before = stub.stub_allocations()
    for _ in range(3):
        call()
    assert stub.stub_allocations() == before
    gpunb.irr_close()
    """)
