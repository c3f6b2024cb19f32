"""CPU: what the library's host side asks of the runtime.  libvoxelcore.so runs in
a child process over a runtime without a device (tests/fake_hip.cpp, preloaded):
kernels do not run and device memory is not touched, so sizes that would fill a GPU
are a matter of milliseconds, and launches, waits and allocations can be counted."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROLOGUE = """
import ctypes, os, sys, threading, time
import numpy as np
sys.path.insert(0, %r)
import voxel_ma_amd as V
F = ctypes.CDLL(os.environ["FAKE_HIP"])
F.fake_items.restype = F.fake_launches.restype = ctypes.c_ulonglong
F.fake_allocs.restype = F.fake_frees.restype = ctypes.c_ulonglong
F.fake_biggest.restype = F.fake_racing.restype = ctypes.c_char_p
F.fake_used.restype = ctypes.c_size_t
F.fake_limit.argtypes = [ctypes.c_size_t]
F.fake_read.argtypes = [ctypes.c_uint32]
P = lambda a: a.ctypes.data_as(ctypes.c_void_p)
vc = V.Context(0)
L = vc._lib
F.fake_reset()
""" % ROOT


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wall",
                    "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", lib, "-lpthread"],
                   check=True)

    def run(body, timeout=120):
        env = dict(os.environ)
        pre = env.get("LD_PRELOAD", "")
        env["LD_PRELOAD"] = lib + (":" + pre if pre else "")
        env["FAKE_HIP"] = lib
        r = subprocess.run([sys.executable, "-c", PROLOGUE + textwrap.dedent(body)], cwd=ROOT,
                           env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                           timeout=timeout)
        assert r.returncode == 0, r.stdout[-4000:]
    return run


@pytest.mark.parametrize("case", ["sides", "faces", "triangles"])
def test_launches_below_the_dispatch_limit(fake, case):
    """A launch holds fewer than 2^32 work-items along an axis.  The pair table of
    2^29 sides has 2^31 slots of two words; 2^30 faces have four lanes each."""
    fake("""
    case = %r
    ne = ctypes.c_int()
    if case == "triangles":  # the counts are read from the device
        n = 4
        fo, fv = np.arange(0, 3 * n + 1, 3, dtype=np.int64), np.zeros(3 * n, np.int32)
        val, lam = np.ones(1, np.uint8), np.zeros(n, np.float32)
        c = [ctypes.c_int64() for _ in range(3)]
        for v in (1, 0, (1 << 29) // 3 + 1):
            F.fake_read(v)
        out = np.zeros(3, np.int32)
        rc = L.vc_voro_extract_inside_device(
            vc.handle, 1, 0, n, None, P(fo), P(fv), P(val), None, P(lam), None, 0,
            ctypes.byref(c[0]), None, None, 0, ctypes.byref(c[1]), P(out), None, None, 1,
            ctypes.byref(c[2]))
        assert rc == V.VC_ERR_CAPACITY and c[2].value == (1 << 29) // 3 + 1
    else:
        nf, nfv = (1, 1 << 29) if case == "sides" else (1 << 30, 0)
        fo = np.zeros(nf + 1, np.int64)
        fo[nf] = nfv
        fv = np.zeros(max(nfv, 1), np.int32)
        vc.check(L.vc_cc_finalize_device(vc.handle, 1, 0, None, nf, P(fo), P(fv), None, 0,
                                         ctypes.byref(ne), P(fv)))
    assert F.fake_launches() > 0
    assert F.fake_items() < 1 << 32, (F.fake_items(), F.fake_biggest())
    """ % case)


def test_allocations_go_on_while_another_context_frees(fake):
    """hipFree waits for its device: a context whose blocks are too large to be
    kept (4.6 GB here) frees them on a busy device, and another context's
    allocations from its own kept blocks do not wait for it."""
    fake("""
    shape = (1024, 1024, 1100)
    other = V.Context(0)
    warm = lambda: other.upload(np.ones((20, 20, 20), np.uint8)).release()
    warm()
    big = vc.from_device(4096, shape).edt()
    F.fake_hold(1)
    a = threading.Thread(target=big.release)
    b = threading.Thread(target=warm)
    a.start()
    while not F.fake_held():
        time.sleep(0.01)
    n = F.fake_allocs()
    b.start()
    b.join(10)
    waited = b.is_alive()
    F.fake_hold(0)
    a.join()
    b.join()
    assert not waited and F.fake_allocs() == n
    """)
