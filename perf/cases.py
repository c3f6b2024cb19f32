"""The calls whose speed is measured: volumes through the framework's public
entry points, at the sizes and on the kinds of shape that they are used on.

  skeleton  a volume resident in device memory: squared distance and feature
            transform, medial measure, thinning at three thresholds (what
            `voroUtility -md=vol2skel` computes per volume)
  serve     the same in one call that allocates nothing, for a serving loop
  oneshot   the same from host bytes to host labels, the volume made and
            released by the call
  edt       the distance and feature transform alone, on a thick solid
  batch     many volumes of uneven sizes, one launch per pass over all
  mesh      boundary sites, quads and Euler terms of a new volume
            (`-md=vol2mesh`), into host arrays
  core      the discrete Voronoi diagram, its inside part and the collapse at
            one threshold (`-md=vol2ma`), into host arrays
  infer     the learned measure of every voxel, into host arrays
  train     loss and weight gradients of the learned measure on one volume
  guided    the pipeline with the gated learned measure in place of the exact

Every volume is made from its case and seed: blurred Gaussian noise, unions
of balls and tori, or one thick ellipsoid.
"""
import ctypes
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

import voxel_ma_amd as V
from voxel_ma_amd import surrogate, synth

_TT = (0.01, 0.02, 0.04)  # thresholds as fractions of the inside size


def listed():
    return [
        # one small part per request in a serving loop: launches and waits
        {"name": "serve 64^3 solids", "kind": "serve", "nx": 64, "ny": 64, "nz": 64},
        # a scanned part given as host bytes, the skeleton wanted back once
        {"name": "oneshot 96x81x107 solids", "kind": "oneshot", "nx": 96, "ny": 81, "nz": 107},
        # an ordinary volume of separate and touching balls
        {"name": "skeleton 256^3 balls", "kind": "skeleton", "shape": "balls",
         "nx": 256, "ny": 256, "nz": 256, "sigma": 0.0},
        # a cropped scan: no axis a multiple of a tile, a word or 8 voxels
        {"name": "skeleton 301x222x437 noise", "kind": "skeleton", "shape": "noise",
         "nx": 301, "ny": 222, "nz": 437, "sigma": 8.0},
        # the benchmark's volume: a porous medium at full size
        {"name": "skeleton 512^3 noise", "kind": "skeleton", "shape": "noise",
         "nx": 512, "ny": 512, "nz": 512, "sigma": 12.0},
        # distances and sites inside a solid that fills the grid (deep voxels)
        {"name": "edt 512^3 ball", "kind": "edt", "nx": 512, "ny": 512, "nz": 512},
        # a shelf of parts of uneven sizes processed together
        {"name": "batch 64 solids", "kind": "batch", "count": 64, "lmin": 32, "lmax": 192},
        # the boundary mesh of a porous medium
        {"name": "mesh 256^3 noise", "kind": "mesh", "nx": 256, "ny": 256, "nz": 256,
         "sigma": 8.0},
        # the medial complex of a small porous block
        {"name": "core 96^3 noise", "kind": "core", "nx": 96, "ny": 96, "nz": 96, "sigma": 8.0},
        # the network alone on a cropped scan (padded to multiples of 8)
        {"name": "infer 150x131x164 noise", "kind": "infer", "nx": 150, "ny": 131, "nz": 164,
         "sigma": 8.0},
        # one volume of a training step at the size the weights were trained on
        {"name": "train 128^3 solids", "kind": "train", "nx": 128, "ny": 128, "nz": 128},
        # the guided pipeline at full size
        {"name": "guided 512^3 noise", "kind": "guided", "nx": 512, "ny": 512, "nz": 512,
         "sigma": 12.0},
    ]


def draw(rng):
    kind = rng.choice(("serve", "oneshot", "skeleton", "skeleton", "edt", "batch", "mesh", "core",
                       "infer", "train", "guided"))

    def axis(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def dims(lo, hi):
        return {"nx": axis(lo, hi), "ny": axis(lo, hi), "nz": axis(lo, hi)}

    def sigma():
        return round(rng.uniform(4.0, 12.0), 2)

    if kind == "serve":
        return dict(kind=kind, **dims(24, 160))
    if kind == "oneshot":
        return dict(kind=kind, **dims(32, 256))
    if kind == "skeleton":
        return dict(kind=kind, shape=rng.choice(("balls", "noise")), sigma=sigma(),
                    **dims(64, 512))
    if kind == "edt":
        return dict(kind=kind, **dims(64, 512))
    if kind == "batch":
        lo = axis(24, 64)
        return dict(kind=kind, count=axis(4, 64), lmin=lo, lmax=axis(lo + 1, 192))
    if kind == "mesh":
        return dict(kind=kind, sigma=sigma(), **dims(64, 320))
    if kind == "core":
        return dict(kind=kind, sigma=sigma(), **dims(32, 112))
    if kind == "infer":
        return dict(kind=kind, sigma=sigma(), **dims(48, 224))
    if kind == "train":
        return dict(kind=kind, **dims(48, 144))
    return dict(kind=kind, sigma=sigma(), **dims(64, 512))


# ------------------------------------------------------------------ volumes
_kept = {}


def _ctx():
    """One context per program, as the command-line tools and the bench keep."""
    if "ctx" not in _kept:
        _kept["ctx"] = V.Context(0)
    return _kept["ctx"]


def _net():
    """The network with the committed weights, loaded once per program."""
    if "net" not in _kept:
        _kept["net"] = V.Surrogate(_ctx(), seed=1, path=surrogate.WEIGHTS)
    return _kept["net"]


def _untrained():
    """A network at the start of its training: He-uniform weights, small
    biases, the same ones in every pass."""
    if "untrained" not in _kept:
        _kept["untrained"] = V.Surrogate(_ctx(), seed=1)
        _kept["untrained"].set_params(_initial())
    return _kept["untrained"]


def _initial():
    rng = np.random.default_rng(11)
    parts = []
    for ci, co in _LAYERS:
        a = math.sqrt(6.0 / (27 * ci))
        parts += [rng.uniform(-a, a, 27 * ci * co), rng.uniform(0.0, 0.05, co)]
    parts += [rng.uniform(-0.06, 0.06, 32), np.zeros(2)]
    return np.concatenate(parts).astype(np.float32)


def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _shell(occ):
    for a in range(3):
        occ.narrow(a, 0, 1).zero_()
        occ.narrow(a, occ.shape[a] - 1, 1).zero_()
    return occ


def _grids(shape):
    return [torch.arange(n, device="cuda", dtype=torch.float32).reshape(
        [-1 if a == b else 1 for b in range(3)]) for a, n in enumerate(shape)]


def _noise(shape, sigma, seed):
    """Blurred Gaussian noise above its 70th percentile, 1-voxel empty shell."""
    g = torch.Generator(device="cuda").manual_seed(seed * 7 + 1)
    v = torch.randn(shape, device="cuda", generator=g)
    taps = torch.from_numpy(synth.gaussian_taps(sigma)).to("cuda")
    rad = (len(taps) - 1) // 2
    for a in range(3):  # periodic, one axis at a time
        acc = torch.zeros_like(v)
        for t in range(len(taps)):
            acc += taps[t] * torch.roll(v, rad - t, dims=a)
        v = acc
    k = max(1, int(math.ceil(0.7 * v.numel())))
    thr = v.reshape(-1).sort().values[k - 1]
    return _shell((v > thr).to(torch.uint8))


def _balls(shape, seed):
    """32 balls per 256^3 voxels (at least 4), radius 8 to 40 at most a third
    of the shortest axis, in a 4-voxel empty margin."""
    rng = np.random.default_rng(seed)
    n = max(4, round(32 * shape[0] * shape[1] * shape[2] / 256 ** 3))
    hi = max(6, min(40, min(shape) // 3))
    gx, gy, gz = _grids(shape)
    occ = torch.zeros(shape, device="cuda", dtype=torch.bool)
    for _ in range(n):
        r = int(rng.integers(min(8, hi - 1), hi + 1))
        c = [int(rng.integers(min(8, m // 2), max(m - 8, m // 2 + 1))) for m in shape]
        lo = [max(c[a] - r, 0) for a in range(3)]
        sl = tuple(slice(lo[a], min(c[a] + r + 1, shape[a])) for a in range(3))
        occ[sl] |= ((gx[sl[0]] - c[0]) ** 2 + (gy[:, sl[1]] - c[1]) ** 2
                    + (gz[:, :, sl[2]] - c[2]) ** 2) <= r * r
    occ = occ.to(torch.uint8)
    for a in range(3):
        occ.narrow(a, 0, 4).zero_()
        occ.narrow(a, shape[a] - 4, 4).zero_()
    return occ


def _solids(shape, seed):
    """Tori and balls in the style of the training volumes, scaled per axis."""
    rng = np.random.default_rng(seed)
    g = [2.0 * x / (n - 1) - 1.0 for x, n in zip(_grids(shape), shape)]  # [-1, 1]
    occ = torch.zeros(shape, device="cuda", dtype=torch.bool)
    for _ in range(int(rng.integers(4, 13))):
        c = rng.uniform(-0.6, 0.6, 3)
        d = [x - float(v) for x, v in zip(g, c)]
        if rng.random() < 0.5:
            R, r = rng.uniform(0.25, 0.6), rng.uniform(0.1, 0.22)
            a, b, e = np.roll([0, 1, 2], int(rng.integers(3)))
            rho = torch.sqrt(d[a] ** 2 + d[b] ** 2) - float(R)
            occ |= (rho ** 2 + d[e] ** 2) <= float(r * r)
        else:
            r = float(rng.uniform(0.12, 0.5))
            occ |= (d[0] ** 2 + d[1] ** 2 + d[2] ** 2) <= r * r
    return _shell(occ.to(torch.uint8))


def _thick(shape, seed):
    """One ellipsoid that nearly fills the grid."""
    rng = np.random.default_rng(seed)
    q = 0.0
    for x, n in zip(_grids(shape), shape):
        q = q + ((x - float((n - 1) / 2 + rng.uniform(-0.01, 0.01) * n))
                 / float(rng.uniform(0.47, 0.49) * n)) ** 2
    return _shell((q <= 1.0).to(torch.uint8))


def _occupancy(case, seed):
    shape, kind = _dims(case), case["kind"]
    if kind == "edt":
        return _thick(shape, seed)
    if kind in ("serve", "oneshot", "train"):
        return _solids(shape, seed)
    if case.get("shape") == "balls":
        return _balls(shape, seed)
    return _noise(shape, case["sigma"], seed)


def _levels(occ):
    size = 0
    for a in range(3):
        idx = occ.amax(dim=[b for b in range(3) if b != a]).nonzero()
        size = max(size, int(idx[-1] - idx[0]) if len(idx) else 0)
    return np.array(synth.levels_from_tt(np.float32(max(size, 1)), _TT), np.float32)


def _volume(occ):
    torch.cuda.synchronize()  # the context has a stream of its own
    vol = _ctx().from_device(occ.data_ptr(), tuple(occ.shape))
    _ctx().synchronize()
    return vol


# ---------------------------------------------------------------- preparing
def _batch_members(case, seed):
    """Edges spread over [lmin, lmax] by their logarithm, always the same ones
    of a case; the solids in them from the seed."""
    n, lo, hi = case["count"], case["lmin"], case["lmax"]
    edges = np.round(lo * (hi / lo) ** ((np.arange(n) + 0.5) / n)).astype(int)
    edges = np.random.default_rng(n).permutation(edges)
    return [_solids((int(e),) * 3, seed * 1009 + i) for i, e in enumerate(edges)]


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "batch":
        occs = _batch_members(case, seed)
        s["levels"] = np.stack([_levels(o) for o in occs])
        s["vols"] = [_volume(o) for o in occs]
        s["batch"] = V.Batch(_ctx(), s["vols"])
        ends = np.cumsum([0] + [o.numel() for o in occs])
        s["label"] = torch.empty(int(ends[-1]), device="cuda", dtype=torch.uint8)
        s["at"] = [(int(a), int(b - a)) for a, b in zip(ends, ends[1:])]
        return s
    occ = _occupancy(case, seed)
    if kind in ("serve", "oneshot", "skeleton", "core", "guided"):
        s["levels"] = _levels(occ)
    if kind == "oneshot":
        s["occ"] = occ.cpu().numpy()
        return s
    if kind in ("serve", "mesh"):
        s["occ"] = occ
        torch.cuda.synchronize()
    else:
        s["vol"] = _volume(occ)
    if kind in ("serve", "skeleton", "guided"):
        s["label"] = torch.empty(_dims(case), device="cuda", dtype=torch.uint8)
    if kind in ("skeleton", "edt"):
        s["edt"] = torch.empty(_dims(case), device="cuda", dtype=torch.int32)
    if kind == "edt":
        s["ft"] = torch.empty(_dims(case), device="cuda", dtype=torch.int32)
    if kind == "train":
        s["vol"].edt().measure()
        _untrained()
    if kind in ("infer", "guided"):
        _net()
    # host arrays as a program that handles many volumes keeps them, large
    # enough for any volume of the case: their filled part is the result
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "mesh":
        cap = int(1.5 * n / case["sigma"]) + 50000
        s["sites"], s["quads"] = np.zeros((cap, 3), np.float32), np.zeros((cap, 4), np.int32)
    if kind == "core":
        s["inside"] = {"vertices": np.zeros(n, np.int32), "vertex_measure": np.zeros(n, np.float32),
                       "edges": np.zeros((3 * n, 2), np.int32),
                       "edge_measure": np.zeros(3 * n, np.float32),
                       "triangles": np.zeros((2 * n, 3), np.int32),
                       "from_face": np.zeros(2 * n, np.int32),
                       "face_measure": np.zeros(2 * n, np.float32)}
        s["kept"] = {"vertices": np.zeros(n, np.int32), "edges": np.zeros((3 * n, 2), np.int32),
                     "triangles": np.zeros((2 * n, 3), np.int32),
                     "from_face": np.zeros(2 * n, np.int32)}
    return s


# ------------------------------------------------------------------ running
def _to(vol, which, t):
    vol.get_device(which, t.data_ptr(), t.numel() * t.element_size())
    return t


def run(s):
    return _RUN[s["kind"]](s)


def _serve(s):
    occ, ctx, lv = s["occ"], _ctx(), s["levels"]
    ctx.check(V.library().vc_skeleton_noalloc(
        ctx.handle, occ.data_ptr(), *occ.shape, lv.ctypes.data, len(lv), s["label"].data_ptr(),
        None))
    return s["label"]


def _oneshot(s):
    vol = _ctx().upload(s["occ"])
    vol.edt().measure().thin_levels(s["levels"], stats=False)
    label = vol.get(V.BUF_LABEL)
    vol.release()
    return label


def _skeleton(s):
    vol = s["vol"]
    vol.edt().measure().thin_levels(s["levels"], stats=False)
    # the skeleton's radii are the roots of the squared distances
    return _to(vol, V.BUF_LABEL, s["label"]), _to(vol, V.BUF_EDT, s["edt"])


def _edt(s):
    vol = s["vol"].edt()
    return _to(vol, V.BUF_EDT, s["edt"]), _to(vol, V.BUF_FT, s["ft"])


def _batch(s):
    s["batch"].run(s["levels"], stats=False)
    for vol, (a, n) in zip(s["vols"], s["at"]):
        _to(vol, V.BUF_LABEL, s["label"][a:a + n])
    return s["label"]


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _mesh(s):
    # the boundary is computed once per volume, so a pass makes its volume
    ctx = _ctx()
    vol = ctx.from_device(s["occ"].data_ptr(), tuple(s["occ"].shape))
    ns, nq, euler = ctypes.c_int64(), ctypes.c_int64(), V.Euler()
    ctx.check(V.library().vc_boundary_extract(
        ctx.handle, vol.handle, _ptr(s["sites"]), len(s["sites"]), ctypes.byref(ns),
        _ptr(s["quads"]), len(s["quads"]), ctypes.byref(nq), ctypes.byref(euler)))
    vol.release()
    return s["sites"], s["quads"], ns.value, nq.value, euler.as_dict()


def _core(s):
    ctx, vol, L, a, k = _ctx(), s["vol"].edt(), V.library(), s["inside"], s["kept"]
    vd = V.VoroDiagram(vol).radii().tag(vol)
    vd.merge_close(1e-3, True)
    n = [ctypes.c_int64() for _ in range(6)]
    cc = V.CellComplex.__new__(V.CellComplex)
    cc.ctx, cc.handle = ctx, ctypes.c_void_p()
    ctx.check(L.vc_vdiag_extract_inside(
        ctx.handle, vd.handle, 0, _ptr(a["vertices"]), _ptr(a["vertex_measure"]),
        len(a["vertices"]), ctypes.byref(n[0]), _ptr(a["edges"]), _ptr(a["edge_measure"]),
        len(a["edges"]), ctypes.byref(n[1]), _ptr(a["triangles"]), _ptr(a["from_face"]),
        _ptr(a["face_measure"]), len(a["triangles"]), ctypes.byref(n[2]),
        ctypes.byref(cc.handle)))
    thin = cc.thinning()
    thin.assign(a["edge_measure"], a["face_measure"])
    thin.prune(float(s["levels"][-1]), float(s["levels"][-1]))
    ctx.check(L.vc_ccthin_remaining(
        ctx.handle, thin.handle, _ptr(k["vertices"]), len(k["vertices"]), ctypes.byref(n[3]),
        _ptr(k["edges"]), len(k["edges"]), ctypes.byref(n[4]), _ptr(k["triangles"]),
        _ptr(k["from_face"]), len(k["triangles"]), ctypes.byref(n[5])))
    thin.release()
    cc.release()
    vd.release()
    return {"inside": a, "kept": k, "counts": [x.value for x in n]}


def _infer(s):
    lam, rel = _net().infer(s["vol"].edt())
    return {"lambda": lam, "relerr": rel}


def _train(s):
    loss, grads = _untrained().gradients(s["vol"])
    return {"loss": loss, "grads": grads}


def _guided(s):
    vol = s["vol"].edt()
    _net().measure(vol, max_rel_err=0.01)
    vol.thin_levels(s["levels"], stats=False)
    return _to(vol, V.BUF_LABEL, s["label"])


_RUN = {"serve": _serve, "oneshot": _oneshot, "skeleton": _skeleton, "edt": _edt, "batch": _batch,
        "mesh": _mesh, "core": _core, "infer": _infer, "train": _train, "guided": _guided}


# --------------------------------------------------------- work, tolerance
_FLOP = 116e3  # of the network's forward pass per voxel


def work(case):
    kind = case["kind"]
    if kind == "batch":
        n, lo, hi = case["count"], case["lmin"], case["lmax"]
        edges = np.round(lo * (hi / lo) ** ((np.arange(n) + 0.5) / n))
        return {"bytes": 2.0 * float((edges ** 3).sum()), "flops": 0.0}
    n = float(case["nx"]) * case["ny"] * case["nz"]
    pad = float(np.prod([(a + 7) // 8 * 8 for a in _dims(case)]))
    if kind in ("serve", "oneshot"):  # occupancy in, labels out
        return {"bytes": 2 * n, "flops": 0.0}
    if kind == "skeleton":  # and the squared distances
        return {"bytes": 6 * n, "flops": 0.0}
    if kind == "edt":  # occupancy in, distances and features out
        return {"bytes": 9 * n, "flops": 0.0}
    if kind == "mesh":  # 12 bytes a site, 16 a quad, about 0.62 / sigma of each a voxel
        return {"bytes": n * (1 + 28 * 0.62 / case["sigma"]), "flops": 0.0}
    if kind == "core":  # about 0.43 faces a voxel, of 2 triangles (20 bytes), 5 sides (12)
        return {"bytes": n * (1 + 0.43 * (2 * 20 + 5 * 12 + 8)), "flops": 0.0}
    if kind == "infer":  # occupancy in, two floats out
        return {"bytes": 9 * n, "flops": _FLOP * pad}
    if kind == "train":  # the backward pass is two forward passes' products
        return {"bytes": 9 * n, "flops": 3 * _FLOP * pad}
    return {"bytes": 2 * n, "flops": _FLOP * pad}


def tolerance(case):
    kind = case["kind"]
    # bf16 weights and activations (and their gradients) through 14 layers: the
    # same rounding points with sums in 64 and in 32 bits differ by up to rel
    # 0.0037, max 0.052 (outputs) and rel 0.0047, max 0.19 (gradients)
    if kind == "infer":
        return {"rel": 0.015, "max": 0.2}
    if kind == "train":
        return {"rel": 0.02, "max": 0.8}
    if kind == "guided":  # a measure at a threshold or at the gate may fall either way
        return {"rel": 0.0, "differ": 0.0001}
    # integer and correctly rounded work with one defined answer
    return "exact"


# ------------------------------------------------- the network in 64 bits
_LAYERS = ((2, 16), (16, 16), (16, 32), (32, 32), (32, 48), (48, 48), (48, 64), (64, 64),
           (112, 48), (48, 48), (80, 32), (32, 32), (48, 16), (16, 16))
_TAPS = [(x, y, z) for x in range(3) for y in range(3) for z in range(3)]


def _weights():
    with open(surrogate.WEIGHTS, "rb") as f:
        f.read(16)  # magic, count
        return np.frombuffer(f.read(), np.float32)


def _features(occ):
    """Exact squared distances and the nearest background voxel (the lowest
    index among equals: ascending candidates, replaced by strictly nearer)."""
    d = torch.where(occ > 0, 1e9, 0.0).to(torch.float64)
    ft = []
    for a in (2, 1, 0):
        n = d.shape[a]
        i = torch.arange(n, device="cuda", dtype=torch.float64).reshape(
            [-1 if b == a else 1 for b in range(3)])
        best = torch.full_like(d, 1e10)
        at = torch.zeros(d.shape, device="cuda", dtype=torch.int64)
        for j in range(n):
            c = d.narrow(a, j, 1) + (i - j) ** 2
            less = c < best
            best = torch.where(less, c, best)
            at = torch.where(less, j, at)
        d = best
        ft = [at] + [f.gather(a, at) for f in ft]
    return d, ft


def _lam2(occ, ft):
    """Largest squared distance between the features of a voxel and of its
    inside 6-neighbours; 0 outside."""
    lam = torch.zeros(occ.shape, device="cuda", dtype=torch.int64)
    for a in range(3):
        n = occ.shape[a] - 1
        both = (occ.narrow(a, 0, n) > 0) & (occ.narrow(a, 1, n) > 0)
        d2 = sum((f.narrow(a, 0, n) - f.narrow(a, 1, n)) ** 2 for f in ft)
        d2 = torch.where(both, d2, 0)
        for at in (0, 1):
            v = lam.narrow(a, at, n)
            v.copy_(torch.maximum(v, d2))
    return lam


def _conv(x, w, b):
    X, Y, Z, _ = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b.expand(X, Y, Z, -1)
    for t, (i, j, k) in enumerate(_TAPS):
        out = out + p[i:i + X, j:j + Y, k:k + Z].reshape(X * Y * Z, -1).matmul(w[t]).reshape(
            X, Y, Z, -1)
    return torch.relu(out)


def _pool(x):
    X, Y, Z, C = x.shape
    return x.reshape(X // 2, 2, Y // 2, 2, Z // 2, 2, C).mean(dim=(1, 3, 5))


def _up(x):
    for a in range(3):
        x = x.repeat_interleave(2, dim=a)
    return x


def _unet(theta, occ, edt):
    """The two outputs of every voxel of the padded volume."""
    parts, o = [], 0
    for ci, co in _LAYERS:
        n = 27 * ci * co
        parts.append((theta[o:o + n].reshape(27, ci, co), theta[o + n:o + n + co]))
        o += n + co
    grow = [(-m) % 8 for m in occ.shape]
    pad = (0, grow[2], 0, grow[1], 0, grow[0])
    x = torch.stack([torch.nn.functional.pad((occ > 0).double(), pad),
                     torch.nn.functional.pad(edt.sqrt() / 32.0, pad)], dim=3)

    def two(x, i):
        for k in (i, i + 1):
            x = checkpoint(_conv, x, *parts[k], use_reentrant=False)
        return x
    skips = []
    for i in (0, 2, 4):
        x = two(x, i)
        skips.append(x)
        x = _pool(x)
    x = two(x, 6)
    for i in (8, 10, 12):
        x = two(torch.cat([_up(x), skips.pop()], dim=3), i)
    return x.matmul(theta[o:o + 32].reshape(16, 2)) + theta[o + 32:o + 34]


def exact(case, seed):
    """The network's outputs, loss and gradients in 64 bits; the other kinds
    return whole numbers, or measures that are exact roots of them."""
    if case["kind"] not in ("infer", "train"):
        return None
    occ = _occupancy(case, seed)
    nx, ny, nz = occ.shape
    theta = _weights() if case["kind"] == "infer" else _initial()
    theta = torch.from_numpy(theta.astype(np.float64)).to("cuda")
    edt, ft = _features(occ)
    if case["kind"] == "infer":
        with torch.no_grad():
            out = _unet(theta, occ, edt)[:nx, :ny, :nz]
        return {"lambda": (out[..., 0] * 32.0).cpu(), "relerr": out[..., 1].exp().cpu()}
    theta.requires_grad_(True)
    out = _unet(theta, occ, edt)[:nx, :ny, :nz]
    t = _lam2(occ, ft).double().sqrt() / 32.0
    r = (out[..., 0] - t) / (t + 1.0 / 32.0)
    e = torch.log(r.detach().abs() + 1e-4)
    inside = occ > 0
    loss = (torch.where(inside, r * r + 0.1 * (out[..., 1] - e) ** 2, 0.0).sum()
            / max(int(inside.sum()), 1))
    loss.backward()
    return {"loss": float(loss.detach()), "grads": theta.grad.cpu()}

