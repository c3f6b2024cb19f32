"""GPU: the memory that a context frees and hands out again.  Volumes of sizes
that share and miss each other's blocks, made and released in turn (a release
waits for the context's stream) in two threads with a context each: every result
equals the oracle's; a context can be destroyed and another made in between.
Scratch that is freed and handed out while queued work still runs, on either
stream.  Memory given back to the device.  (The bounds of what is kept are tested
without a device, in test_host_side.py.)"""
import ctypes
import threading

import numpy as np
import pytest

import voxel_ma_amd as V
from conftest import say

pytestmark = pytest.mark.gpu

SHAPES = [(20, 20, 20), (21, 20, 20), (40, 33, 70), (8, 8, 8), (64, 40, 24), (20, 20, 21)]


@pytest.mark.parametrize("threads", [1, 2])
def test_reused_blocks(oracle, threads):
    rng = np.random.default_rng(41)
    levels = [1.0, 2.5]
    cases = []
    for shape in SHAPES:
        occ = (rng.random(shape) < 0.85).astype(np.uint8)
        d, f = oracle.edt_ft(occ)
        lvl = oracle.levels(occ, oracle.lambda2(occ, f), levels)
        cases.append((occ, d, oracle.thin(occ, lvl, len(levels))[0]))
    say("reused blocks", threads, "threads")
    wrong = []

    def work(seed):
        order = np.random.default_rng(seed).integers(0, len(cases), 60)
        ctx = V.Context(0)
        held = []
        for n, i in enumerate(order):
            occ, d, lab = cases[i]
            vol = ctx.upload(occ)
            vol.edt().measure().thin_levels(levels, stats=False)
            out = V.DeviceBuffer(occ.size)
            vol.get_device(V.BUF_LABEL, out.ptr, out.nbytes)
            if n % 3 == 0:  # some volumes outlive others
                held.append((vol, d))
            else:
                vol.release()
            if len(held) > 4:
                v, dd = held.pop(0)
                if not np.array_equal(v.get(V.BUF_EDT), dd):
                    wrong.append(("edt", n))
                v.release()
            ctx.synchronize()
            if not np.array_equal(out.download(np.uint8, occ.shape), lab):
                wrong.append(("label", n))
            out.free()
            if n == 30:  # a second context's memory is its own
                other = V.Context(0)
                v2 = other.upload(occ)
                v2.edt()
                if not np.array_equal(v2.get(V.BUF_EDT), d):
                    wrong.append(("other", n))
                v2.release()
                other.close()
        for v, _ in held:
            v.release()
        ctx.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 7), (4, 4, 16), (17, 19, 23), (64, 64, 65),
                                   (160, 330, 330)])
def test_results_into_caller_memory(vc, shape):
    """vc_get_device against vc_get for every buffer (features are converted by a
    kernel, the others copied), small and large, and into memory at odd offsets of
    the caller's."""
    rng = np.random.default_rng(5)
    occ = (rng.random(shape) < 0.7).astype(np.uint8)
    vol = vc.upload(occ)
    vol.edt().measure().thin_levels([1.0, 2.0], stats=False)
    N = occ.size
    for which in (V.BUF_OCC, V.BUF_EDT, V.BUF_FT, V.BUF_LAM2, V.BUF_LABEL, V.BUF_LEVEL):
        ref = vol.get(which)
        step = ref.itemsize
        for off in (0, step, 3 * step):
            buf = V.DeviceBuffer.from_array(np.full(N * step + 8 * step, 0xA5, np.uint8))
            say("into caller memory", shape, which, off)
            vol.get_device(which, buf.ptr + off, N * step)
            vc.synchronize()
            out = buf.download(np.uint8, N * step + 8 * step)
            buf.free()
            assert np.array_equal(out[off:off + N * step], ref.reshape(-1).view(np.uint8))
            assert (out[:off] == 0xA5).all() and (out[off + N * step:] == 0xA5).all()
    vol.release()


def test_scratch_grows_behind_queued_work(oracle):
    """The boundary's scratch slots are freed and allocated anew when a larger volume
    comes, without a wait for work queued before: here the transform, measure and
    thinning of another volume, and buffers freed by a third.  The Euler terms run
    on the second stream (rows of a multiple of 8 voxels) or on the first."""
    rng = np.random.default_rng(57)
    ctx = V.Context(0)
    levels = [1.0, 2.5]

    def volume(shape, p=0.85):
        return (rng.random(shape) < p).astype(np.uint8)
    for shapes in ([(9, 10, 8), (17, 16, 24), (40, 33, 48), (64, 50, 72)],
                   [(7, 9, 11), (20, 17, 31), (45, 40, 61), (70, 52, 77)]):
        held = []
        for shape in shapes:
            say("scratch grows", shape)
            occ, bnd = volume((48, 40, 70)), volume(shape, 0.6)
            dead = ctx.upload(volume(shape))
            dead.edt()
            vol, small = ctx.upload(occ), ctx.upload(bnd)
            vol.edt().measure().thin_levels(levels, stats=False)
            dead.release()
            vol.thin_levels(levels, stats=False)
            vol.edt()
            s, q, e = small.boundary()
            held.append((occ, vol, bnd, small, s, q, e))
        for occ, vol, bnd, small, s, q, e in held:
            d, f = oracle.edt_ft(occ)
            lvl = oracle.levels(occ, oracle.lambda2(occ, f), levels)
            assert np.array_equal(vol.get(V.BUF_EDT), d)
            assert np.array_equal(vol.get(V.BUF_LABEL), oracle.thin(occ, lvl, len(levels))[0])
            so, qo, eo = oracle.boundary(bnd)
            assert np.array_equal(s, so) and np.array_equal(q, qo)
            assert e["euler"] == eo["euler"] and e["C"] == eo["C"]
            assert e["chi"] == oracle.euler_voxels(bnd)
            vol.release()
            small.release()
    ctx.close()


def test_trim_gives_memory_back(oracle):
    """A released volume's 400 MB stay with the context until vc_ctx_trim; the next
    volume is right with and without them."""
    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert V.hip().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value
    rng = np.random.default_rng(3)
    small = (rng.random((30, 31, 33)) < 0.8).astype(np.uint8)
    ref = oracle.edt_ft(small)[0]
    ctx = V.Context(0)
    for trim in (False, True, True):
        before = free()
        vol = ctx.upload(np.ones((300, 300, 300), np.uint8))
        vol.edt().measure().thin_levels([1.0], stats=False)
        vol.release()
        kept = free()
        say("trim", before, kept)
        if trim:
            ctx.trim()
            assert free() > kept + (300 << 20)
        vol = ctx.upload(small)
        vol.edt()
        assert np.array_equal(vol.get(V.BUF_EDT), ref)
        vol.release()
    ctx.close()
