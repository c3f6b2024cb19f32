"""GPU parity: measure-ordered subfield thinning through the C ABI against the
CPU oracle's dense schedule (bit-exact labels) plus topology invariants."""
import itertools

import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu


def _gpu_thin(vc, occ, levels):
    vol = vc.upload(occ)
    vol.edt().measure()
    st = vol.thin_levels(levels)
    lab, lvl = vol.get(4), vol.get(5)
    vol.release()
    return lab, lvl, st


def _oracle_thin(oracle, occ, levels):
    d, f = oracle.edt_ft(occ)
    lam = oracle.lambda2(occ, f)
    lvl = oracle.levels(occ, lam, levels)
    lab, st = oracle.thin(occ, lvl, len(levels))
    return lab, lvl, st


def _compare(vc, oracle, occ, levels, name):
    say("thin", name, occ.shape, levels)
    lab, lvl, st = _gpu_thin(vc, occ, levels)
    labo, lvlo, sto = _oracle_thin(oracle, occ, levels)
    assert np.array_equal(lvl, lvlo), name
    assert np.array_equal(lab, labo), name
    for k in range(len(levels)):
        assert st.removed[k] == sto.removed[k]
    # the same number of sweeps as the dense schedule (8 passes per sweep)
    assert st.passes == 8 * sum(sto.sweeps[k] for k in range(len(levels)))
    return lab


def test_thin_random_small(vc, oracle):
    rng = np.random.default_rng(9)
    for i in range(25):
        shape = tuple(int(s) for s in rng.integers(2, 30, size=3))
        occ = (rng.random(shape) < rng.choice([0.5, 0.8, 0.95])).astype(np.uint8)
        levels = sorted(float(x) for x in rng.uniform(0.5, 8.0, size=int(rng.integers(1, 5))))
        _compare(vc, oracle, occ, levels, "rand%d" % i)


def test_thin_config1_torus(vc, oracle):
    from voxel_ma_amd import synth
    occ = synth.torus_c1()
    for levels in ([1.5, 3.0, 6.0], synth.levels_from_tt(synth.inside_size(occ), (0.04,))):
        lab = _compare(vc, oracle, occ, levels, "c1")
        b = oracle.betti(occ)
        for k in range(len(levels)):
            assert oracle.betti(((lab == 1) | (lab > 2 + k)).astype(np.uint8)) == b


def test_thin_config2_spheres(vc, oracle):
    from voxel_ma_amd import synth
    occ = synth.spheres_c2()
    levels = synth.levels_from_tt(synth.inside_size(occ))
    lab = _compare(vc, oracle, occ, levels, "c2")
    b = oracle.betti(occ)
    sk = ((lab == 1) | (lab > 2 + len(levels) - 1)).astype(np.uint8)
    assert oracle.betti(sk) == b


def test_thin_float_measure_path(vc, oracle):
    """vc_set_measure_f32: the thinning uses the caller's float measure."""
    import voxel_ma_amd
    from voxel_ma_amd import synth
    occ = synth.torus_c1()
    rng = np.random.default_rng(3)
    meas = rng.uniform(0, 5, size=occ.shape).astype(np.float32)
    levels = [1.0, 2.5, 4.0]
    say("thin float measure")
    vol = vc.upload(occ)
    dm = voxel_ma_amd.DeviceBuffer.from_array(meas)
    vol.set_measure_f32(dm.ptr)
    vol.thin_levels(levels)
    lab, lvl = vol.get(4), vol.get(5)
    vol.release()
    dm.free()
    lvlo = np.full(occ.shape, 255, np.uint8)
    for k in reversed(range(len(levels))):
        lvlo[(occ > 0) & (meas < np.float32(levels[k]))] = k
    assert np.array_equal(lvl, lvlo)
    labo, _ = oracle.thin(occ, lvlo, len(levels))
    assert np.array_equal(lab, labo)


def test_thin_empty_and_full(vc, oracle):
    for name, occ in {"empty": np.zeros((9, 9, 9), np.uint8),
                      "full": np.ones((9, 9, 9), np.uint8),
                      "one": np.pad(np.ones((1, 1, 1), np.uint8), 2)}.items():
        _compare(vc, oracle, occ, [2.0, 5.0], name)


@pytest.mark.parametrize("case", ["ring", "levels", "unwaited"])
def test_thin_watched_levels(vc, oracle, case):
    """The host follows a level through one word that each sweep writes for the
    sweep before it: more sweeps in a level than the device's ring of flags has
    entries (64), many levels in a row of which most converge in their first
    sweep, and calls that follow each other without a wait."""
    if case == "ring":  # a bar loses two voxels per end and sweep
        occ = np.zeros((5, 6, 410), np.uint8)
        occ[2, 3, 3:-3] = 1
        _compare(vc, oracle, occ, [1e6], case)
        occ[1:3, 2:4, 3:-3] = 1
        _compare(vc, oracle, occ, [1.5, 1e6], case)
    elif case == "levels":
        rng = np.random.default_rng(17)
        occ = (rng.random((33, 20, 70)) < 0.9).astype(np.uint8)
        _compare(vc, oracle, occ, [0.25 * q for q in range(64)], case)
    else:
        rng = np.random.default_rng(18)
        occ = (rng.random((40, 37, 50)) < 0.85).astype(np.uint8)
        sets = [[1.5], [0.5, 2.5, 4.0], [1e6]]
        vol = vc.upload(occ)
        vol.edt().measure()
        for levels in sets + sets[::-1]:
            say("thin", case, levels)
            vol.thin_levels(levels, stats=False)
            vol.thin_levels(levels, stats=False)
            assert np.array_equal(vol.get(4), _oracle_thin(oracle, occ, levels)[0])
        vol.release()


@pytest.mark.parametrize("nz", [40, 65, 90, 115, 140])
def test_timed_sweeps_are_those_that_run(vc, nz):
    """With timing on, a level runs as without: launched ahead of the sweeps' own
    reports, with at most three sweeps past the last report (a bar loses two voxels
    per end and sweep; segments between checks would launch up to 15 too many)."""
    import voxel_ma_amd as V
    occ = np.zeros((5, 6, nz), np.uint8)
    occ[2, 3, 3:-3] = 1
    vol = vc.upload(occ)
    vol.edt().measure()
    ref = vol.thin_levels([1e6])
    lab = vol.get(V.BUF_LABEL)
    say("timed sweeps", nz)
    vc.thin_timing(True)
    st = vol.thin_levels([1e6])
    launches, ms = vc.thin_timing_read()
    vol.thin_levels([1e6], stats=False)  # timed calls wait also without statistics
    again, _ = vc.thin_timing_read()
    vc.thin_timing(False)
    sweeps = st.passes // 8
    assert st.passes == ref.passes and st.tests == ref.tests
    assert np.array_equal(vol.get(V.BUF_LABEL), lab)
    assert st.launches == launches + 1 and ms > 0.0  # and the level's set-up
    assert sweeps < launches <= sweeps + 3, (sweeps, launches)
    assert launches + sweeps < again <= launches + sweeps + 3
    vol.release()


@pytest.mark.parametrize("nz", [1, 2, 7, 8, 9, 15, 63, 64, 65, 71, 128, 131, 255, 257, 519])
def test_row_lengths(vc, oracle, nz):
    """Rows of every alignment: the row pass of the EDT and the level set-ups
    read 8 voxels per access, a chunk that the row's end cuts as the row's last
    8 (rows shorter than 8 voxel by voxel), and share a wavefront between short
    rows; the last voxels of a row, inside and outside, and the exact and the
    float measure, against the oracle."""
    import voxel_ma_amd as V
    rng = np.random.default_rng(nz)
    occ = (rng.random((7, 9, nz)) < 0.8).astype(np.uint8)
    occ[3, :, -3:] = 1
    occ[4, :, -3:] = 0
    levels = [0.5, 1.5, 3.0]
    _compare(vc, oracle, occ, levels, "nz %d" % nz)
    vol = vc.upload(occ)
    vol.edt()
    d, f = oracle.edt_ft(occ)
    assert np.array_equal(vol.get(V.BUF_EDT), d) and np.array_equal(vol.get(V.BUF_FT), f)
    meas = rng.uniform(0, 4, size=occ.shape).astype(np.float32)
    dm = V.DeviceBuffer.from_array(meas)
    vol.set_measure_f32(dm.ptr)
    vol.thin_levels(levels)
    lvlo = np.full(occ.shape, 255, np.uint8)
    for k in reversed(range(len(levels))):
        lvlo[(occ > 0) & (meas < np.float32(levels[k]))] = k
    assert np.array_equal(vol.get(V.BUF_LEVEL), lvlo)
    assert np.array_equal(vol.get(V.BUF_LABEL), oracle.thin(occ, lvlo, len(levels))[0])
    vol.release()
    dm.free()
