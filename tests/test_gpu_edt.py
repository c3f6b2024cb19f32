"""GPU parity: EDT, feature transform and measure through the C ABI against
the CPU oracle (bit-exact) and the scipy golden vectors."""
import os

import numpy as np
import pytest

from conftest import say

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.gpu


def _run(vc, occ):
    vol = vc.upload(occ)
    vol.edt().measure()
    d, f, lam = vol.get(1), vol.get(2), vol.get(3)
    vol.release()
    return d, f, lam


def _check(vc, oracle, occ, name):
    say("edt", name, occ.shape)
    d, f, lam = _run(vc, occ)
    do, fo = oracle.edt_ft(occ)
    assert np.array_equal(d, do), name
    assert np.array_equal(f, fo), name
    lo = oracle.lambda2(occ, fo)
    assert np.array_equal(lam.astype(np.int64), lo.astype(np.int64)), name


def test_simple_table_matches_oracle(vc, simple_lut_cpu):
    say("simple table")
    t = vc.simple_table()
    assert np.array_equal(t, simple_lut_cpu)


def test_edt_random_shapes(vc, oracle):
    rng = np.random.default_rng(5)
    for i in range(40):
        shape = tuple(int(s) for s in rng.integers(1, 40, size=3))
        occ = (rng.random(shape) < rng.choice([0.3, 0.7, 0.95, 0.995])).astype(np.uint8)
        _check(vc, oracle, occ, "rand%d" % i)


def test_edt_edge_cases(vc, oracle):
    cases = {
        "all_background": np.zeros((7, 8, 9), np.uint8),
        "all_inside": np.ones((7, 8, 9), np.uint8),
        "one_voxel": np.ones((1, 1, 1), np.uint8),
        "line_x": (np.arange(97) % 13 != 0).astype(np.uint8).reshape(97, 1, 1),
        "line_z": (np.arange(300) % 41 != 0).astype(np.uint8).reshape(1, 1, 300),
        "single_bg": np.ones((33, 17, 65), np.uint8),
        "wide_z": np.ones((3, 4, 2000), np.uint8),
    }
    cases["single_bg"][30, 2, 64] = 0
    cases["wide_z"][1, 2, 1234] = 0
    for name, occ in cases.items():
        _check(vc, oracle, occ, name)


def test_edt_scipy_golden(vc):
    z = np.load(os.path.join(HERE, "golden", "edt_scipy.npz"))
    for name in sorted({k.split("__")[0] for k in z.files}):
        say("edt golden", name)
        d, f, _ = _run(vc, z[name + "__occ"])
        assert np.array_equal(d, z[name + "__d2"]), name


def test_edt_config1_torus(vc, oracle):
    from voxel_ma_amd import synth
    _check(vc, oracle, synth.torus_c1(), "c1")


def test_edt_config2_spheres(vc, oracle):
    from voxel_ma_amd import synth
    _check(vc, oracle, synth.spheres_c2(), "c2")


def test_edt_rows_multiple_of_8(vc, oracle):
    """Rows whose length is a multiple of 8 take the 8-voxels-per-lane row
    pass: lengths that are and are not multiples of 64, sparse background
    (searches across words), rows without background, and consecutive rows
    of very different content (the LDS row masks are reused)."""
    rng = np.random.default_rng(17)
    for nz in (8, 16, 24, 64, 72, 136, 520, 1032):
        for fill in (0.5, 0.9, 0.995):
            occ = (rng.random((5, 6, nz)) < fill).astype(np.uint8)
            occ[1, 2, :] = 1          # a row without background
            occ[3, 0, :] = 0          # a row of background only
            occ[4, 5, :] = 1
            occ[4, 5, nz - 1] = 0     # background only at the row's end
            _check(vc, oracle, occ, "z8 %d %.3f" % (nz, fill))


def test_edt_long_axes(vc, oracle):
    """Axes longer than 16384: the y pass falls back from its 24-bit
    offset arithmetic to the plain one (both must give the same result);
    sparse background so searches run long."""
    rng = np.random.default_rng(19)
    for shape in ((2, 3, 16500), (2, 16500, 3), (3, 2, 20000)):
        occ = (rng.random(shape) < 0.999).astype(np.uint8)
        occ[0, 0, 0] = 0
        _check(vc, oracle, occ, "long %s" % (shape,))


def test_edt_thick_solids(vc, oracle):
    """Thick solids: column searches run past their outward stretch of 16
    distances into the block-by-block continuation, in both column passes.
    A ball centred on a voxel corner (many equal-distance nearest
    background voxels: the lowest index must win), an off-centre ellipsoid
    (lopsided searches), a slab, and a block with a few background voxels
    (searches across the whole column)."""
    n = 96
    g = np.arange(n) - (n - 1) / 2.0
    r2 = g[:, None, None] ** 2 + g[None, :, None] ** 2 + g[None, None, :] ** 2
    cases = {"ball": (r2 <= 44.0 ** 2).astype(np.uint8)}
    h = np.arange(n) - 40.0
    e2 = (h[:, None, None] ** 2 + (1.3 * h[None, :, None]) ** 2 +
          (0.7 * h[None, None, :]) ** 2)
    cases["ellipsoid"] = (e2 <= 38.0 ** 2).astype(np.uint8)
    slab = np.zeros((n, n, n), np.uint8)
    slab[2:-2, 2:-2, 20:76] = 1
    cases["slab"] = slab
    rng = np.random.default_rng(23)
    holes = np.ones((80, 90, 100), np.uint8)
    for _ in range(6):
        holes[tuple(int(rng.integers(0, s)) for s in holes.shape)] = 0
    cases["holes"] = holes
    for name, occ in cases.items():
        _check(vc, oracle, occ, "thick " + name)


@pytest.mark.parametrize("n", [7, 8, 9, 15, 16, 63, 64, 65, 128, 135, 511, 512, 513])
def test_edt_thick_columns_of_every_length(vc, n):
    """Divide and conquer over columns of n rows (blocks of 8^k rows, a top level
    of one row from 8^k to 2 8^k - 1): every tile is flagged, since the few
    background voxels are far along z and from most voxels.  The answer is the
    nearest of those, the lowest index among equals."""
    import voxel_ma_amd as V
    from conftest import say
    rng = np.random.default_rng(n)
    for axis in (0, 1):
        shape = [3, 3, 330]
        shape[axis] = n
        for few in (1, 2, 5):
            occ = np.ones(shape, np.uint8)
            at = np.stack([rng.integers(0, m, few) for m in shape[:2]] +
                          [rng.choice([0, 1, 328, 329], few)], 1)
            if few > 2:  # equal distances across the column's middle
                at[:2] = 0
                at[1, axis] = n - 1
            occ[tuple(at.T)] = 0
            at = np.argwhere(occ == 0)  # in index order
            g = np.indices(shape)
            d = np.stack([sum((g[a] - p[a]) ** 2 for a in range(3)) for p in at])
            k = d.argmin(0)  # the first of equals
            say("thick column", shape, few)
            vol = vc.upload(occ)
            for _ in range(2):  # the flags are cleared and set again
                vol.edt()
                assert np.array_equal(vol.get(V.BUF_EDT), d.min(0))
                assert np.array_equal(vol.get(V.BUF_FT),
                                      np.ravel_multi_index(at.T, shape)[k])
            vol.release()
