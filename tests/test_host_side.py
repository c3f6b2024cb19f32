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


def test_kept_memory_is_bounded_and_given_back(fake):
    """What released volumes leave behind: at most 8 GiB, the oldest blocks gone
    first, none above 2 GiB, all of it back on vc_ctx_trim (one context's or every
    context's), when an allocation would fail (the library's own or a
    DeviceBuffer's), and at the context's end; counted by the runtime."""
    fake("""
    GB = 1 << 30
    other = V.Context(0)
    vc.trim(); other.trim()
    base = F.fake_used(0)

    def run(c, shape):
        v = c.from_device(4096, shape).edt()
        v.release()
    # 900 MB of occupancy: 3.6 GB buffers go back at once, the small ones stay
    run(vc, (1000, 1000, 900))
    kept = F.fake_used(0) - base
    assert 0.9 * GB < kept + GB // 8 and kept < 5 * GB, kept
    vc.trim()
    assert F.fake_used(0) == base
    # 240 MB volumes of growing size classes (960 MB buffers): the cap holds
    for n in range(240, 470, 16):
        run(vc, (1000, 1000, n))
        assert F.fake_used(0) - base <= 8 * GB, n
    assert F.fake_used(0) - base > 6 * GB
    # the newest volume's blocks are still there: nothing is allocated for it
    a = F.fake_allocs()
    run(vc, (1000, 1000, n))
    assert F.fake_allocs() == a
    # one context's memory, then every context's
    run(other, (100, 100, 100))
    mine = F.fake_used(0)
    vc.trim()
    assert base < F.fake_used(0) < mine and F.fake_used(0) - base < GB
    run(vc, (300, 300, 300))
    L.vc_ctx_trim(None)
    assert F.fake_used(0) == base
    # an allocation that would fail takes back what every context keeps
    run(vc, (500, 500, 500)); run(other, (500, 500, 500))
    assert F.fake_used(0) - base > 2 * GB
    F.fake_limit(base + 2 * GB)
    v = vc.from_device(4096, (400, 400, 400)).edt()
    F.fake_limit((1 << 63) - 1)
    v.release()
    run(other, (500, 500, 500))
    F.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    F.hipFree.argtypes = [ctypes.c_void_p]
    V._hip = type("Runtime", (), {"h": F})()
    F.fake_limit(base + 2 * GB)
    b = V.DeviceBuffer(2 * GB - 4096)
    assert F.fake_used(0) == base + b.nbytes
    try:
        vc.from_device(4096, (500, 500, 500))
        raise SystemExit("allocated beyond the limit")
    except V.VcError as e:
        assert e.code == V.VC_ERR_NOMEM
    b.free()
    F.fake_limit((1 << 63) - 1)
    # pinned memory, and the end of a context with and without live volumes
    third = V.Context(0)
    at = F.fake_used(0), F.fake_used(1)
    live = third.from_device(4096, (64, 64, 64)).edt()
    run(third, (64, 64, 64))
    assert F.fake_used(0) > at[0] and F.fake_used(1) > at[1]
    run(third, (64, 64, 64))
    live.release()
    third.close()
    other.close()
    vc.close()
    assert F.fake_used(0) == 0 and F.fake_used(1) == 0, (F.fake_used(0), F.fake_used(1))
    """)


def test_noalloc_call_drains_after_an_error(fake):
    """vc_skeleton_noalloc's scratch array is the device's: a call that fails (no
    sweep reports here, since no kernel runs) returns with nothing in flight, as
    one that succeeds does."""
    fake("""
    lv = np.array([1.0, 2.0], np.float32)
    rc = L.vc_skeleton_noalloc(vc.handle, ctypes.c_void_p(4096), 20, 30, 40, P(lv), 2,
                               ctypes.c_void_p(8192), None)
    assert rc == V.VC_ERR_HIP and "report" in vc.last_error(), (rc, vc.last_error())
    assert F.fake_launches() > 3 and F.fake_unwaited() == 0
    """)


def test_null_stream_copies_wait_for_the_context_stream(fake):
    """The context's stream does not order itself with the null stream, so a copy on
    the null stream comes after a wait for every kernel before it."""
    fake("""
    def ok(what):
        assert F.fake_racing() == b"", (what, F.fake_racing())
    occ = np.ones((40, 33, 70), np.uint8)
    vol = vc.upload(occ)
    vol.edt().measure()
    vol.boundary()
    ok("volume")
    for _ in range(2):
        V.Batch(vc, [vol, vc.upload(occ)]).edt().measure()
    ok("batch")
    nv, ne, nf = 8, 5, 2
    vts, edges = np.zeros((nv, 3), np.float32), np.zeros((ne, 2), np.int32)
    fo, fv = np.array([0, 4, 8], np.int64), np.zeros(8, np.int32)
    veo, ve = np.zeros(nv + 1, np.int64), np.zeros(1, np.int32)
    val = np.ones(nv, np.uint8)
    i32 = lambda n: P(np.zeros(n, np.int32))
    n1, n2, on = ctypes.c_int(), ctypes.c_int64(), ctypes.c_int()
    out = [np.zeros(32, np.int64) for _ in range(8)]
    rc = L.vc_voro_merge_close_device(
        vc.handle, nv, ne, nf, P(vts), P(edges), P(fo), P(fv), P(veo), P(ve), P(val),
        ctypes.c_float(0.1), 0, P(out[0]), P(out[1]), ctypes.byref(n1), P(out[2]), P(out[3]),
        P(out[4]), P(out[5]), ctypes.c_int64(16), ctypes.byref(n2), P(out[6]), ctypes.byref(on))
    assert rc == V.VC_OK and on.value == 1
    ok("merge")
    net = V.Surrogate(vc, seed=1)
    net.set_params(net.params())
    net.infer(vol)
    net.set_params(net.params())
    ok("surrogate")
    d = V.VoroDiagram(vol)
    ok("diagram")
    """)
