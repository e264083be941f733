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
