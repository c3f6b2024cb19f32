"""GPU checks of the measure surrogate (include/vc_surrogate.h) against the
float64 restatement oracle/unet_ref.py: initial weights bit-exact, every
layer's activations and every layer's weight gradient within BF16
tolerance, training lowers the loss, tiled inference equals whole-volume
inference bit for bit, and the gated measure drives the exact thinning
(labels equal the oracle's thinning under the same measure)."""
import os
import sys

import numpy as np
import pytest

import voxel_ma_amd as V
from conftest import ROOT, say

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import unet_ref as U  # noqa: E402

pytestmark = pytest.mark.gpu


def _occ(n, seed):
    from voxel_ma_amd import synth
    rng = np.random.default_rng(seed)
    while True:
        occ = synth.solids_host(n, synth.training_specs(n, rng))
        if occ.sum() > 50:
            return occ


def _theta(seed):
    """Initial weights plus small bias noise (keeps ReLUs alive on tiny
    volumes)."""
    th = U.init_params(seed).astype(np.float64)
    rng = np.random.default_rng(seed + 100)
    o = 0
    for _, ci, co in U.LAYERS:
        o += 27 * ci * co
        th[o:o + co] = rng.uniform(0.0, 0.05, size=co)
        o += co
    return th.astype(np.float32)


@pytest.fixture(scope="module")
def small(vc):
    occ = _occ(24, 12)
    vol = vc.upload(occ)
    vol.edt().measure()
    edt, lam2 = vol.get(V.BUF_EDT), vol.get(V.BUF_LAM2)
    yield occ, edt, lam2, vol
    vol.release()


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def test_initial_weights_match_oracle(vc):
    net = V.Surrogate(vc, seed=3)
    assert np.array_equal(net.params(), U.init_params(3))
    net.release()


def test_forward_layers_match_fp64(vc, small):
    occ, edt, lam2, vol = small
    th = _theta(4)
    net = V.Surrogate(vc, seed=4)
    net.set_params(th)
    loss, _ = net.gradients(vol)
    out_ref, acts, _ = U.forward(th.astype(np.float64), U.inputs(occ, edt), keep=True)
    for l, (name, _, co) in enumerate(U.LAYERS):
        ref = acts[name][1]
        got = net.activation(l, ref.shape)
        say("forward", name, _rel(got, ref))
        assert _rel(got, ref) < 0.03, name
    got = net.activation(14, out_ref.shape)
    assert _rel(got, out_ref) < 0.03
    L_ref, _ = U.loss_and_dout(out_ref, occ, lam2)
    assert abs(loss - L_ref) <= 0.05 * abs(L_ref)
    net.release()


def test_gradients_match_fp64(vc, small):
    """Per-layer weight and bias gradients of the BF16 MFMA backward against
    the float64 backward.  The gradient tensors are BF16 (8-bit mantissa),
    so the error grows with the number of layers the gradient crosses: the
    bound is a relative L2 error below 0.2 and a cosine above 0.98 for every
    block (a wrong index, sign or transposition gives cosines far below)."""
    occ, edt, lam2, vol = small
    th = _theta(5)
    net = V.Surrogate(vc, seed=5)
    net.set_params(th)
    _, g = net.gradients(vol)
    _, g_ref = U.gradients(th.astype(np.float64), occ, edt, lam2)
    o = 0
    bad = []
    for name, ci, co in U.LAYERS + [("head", 16, 2)]:
        nw = (1 if name == "head" else 27) * ci * co
        for part, sl in (("W", slice(o, o + nw)), ("b", slice(o + nw, o + nw + co))):
            a, b = g[sl].astype(np.float64), g_ref[sl]
            cos = float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))
            say("grad", name, part, "rel", round(_rel(a, b), 4), "cos", round(cos, 5))
            if not (_rel(a, b) < 0.2 and cos > 0.98):
                bad.append((name, part, _rel(a, b), cos))
        o += nw + co
    assert not bad, bad
    net.release()


def test_layers_and_gradients_match_bf16_oracle(vc, small):
    """Against the oracle's BF16 variant, which rounds to BF16 where the
    kernels store BF16 (weights, activations, pooled tensors, input
    gradients), the kernels differ only by float32 summation order and the
    rare BF16 rounding it flips: every activation within 1 % (measured at
    most 0.4 %), every weight gradient within 4 % relative L2 per layer and
    5 % per tap block (measured at most 2.6 % and 2.9 %; 27 blocks per layer,
    a dropped or misplaced tap leaves its block at 100 %), bias gradients
    within 4 % (at most 2.7 %).  The float64 comparison above needs 20 %."""
    occ, edt, lam2, vol = small
    th = _theta(5)
    net = V.Surrogate(vc, seed=5)
    net.set_params(th)
    _, g = net.gradients(vol)
    thd = th.astype(np.float64)
    out_ref, acts, _ = U.forward(thd, U.inputs(occ, edt), keep=True, bf16=True)
    worst_act = 0.0
    for l, (name, _, co) in enumerate(U.LAYERS):
        ref = acts[name][1]
        r = _rel(net.activation(l, ref.shape), ref)
        worst_act = max(worst_act, r)
        say("bf16 forward", name, round(r, 5))
        assert r < 0.01, (name, r)
    r = _rel(net.activation(14, out_ref.shape), out_ref)
    say("bf16 forward head", round(r, 5))
    assert r < 0.01
    _, g_ref = U.gradients(thd, occ, edt, lam2, bf16=True)
    o = 0
    bad = []
    for name, ci, co in U.LAYERS + [("head", 16, 2)]:
        taps = 1 if name == "head" else 27
        nw = taps * ci * co
        a, b = g[o:o + nw].astype(np.float64), g_ref[o:o + nw]
        rw = _rel(a, b)
        rt = max(_rel(a.reshape(taps, -1)[t], b.reshape(taps, -1)[t]) for t in range(taps))
        rb = _rel(g[o + nw:o + nw + co].astype(np.float64), g_ref[o + nw:o + nw + co])
        say("bf16 grad", name, "W", round(rw, 5), "worst tap", round(rt, 5), "b", round(rb, 5))
        if not (rw < 0.04 and rt < 0.05 and rb < 0.04):
            bad.append((name, rw, rt, rb))
        o += nw + co
    assert not bad, bad
    net.release()


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 24, 40), (23, 9, 66), (96, 88, 8)])
def test_weight_gradients_on_partial_and_chunked_bricks(vc, shape):
    """The weight gradient's bricks are 4 x 4 x 32 voxels: levels with fewer
    voxels than a brick along every axis, a second partly filled brick along z,
    ragged axes, and more bricks than chunks (a workgroup walks several).
    Against the BF16 variant of the oracle with the bounds of
    test_layers_and_gradients_match_bf16_oracle; a dropped brick or a wrong
    edge leaves its layer far outside them."""
    from voxel_ma_amd import synth
    rng = np.random.default_rng(sum(shape))
    L = max(shape)
    occ = np.zeros(shape, np.uint8)
    while occ.sum() < 40:
        o = synth.solids_host(L, synth.training_specs(L, rng)) if L <= 48 else \
            (rng.random((L,) * 3) < 0.6).astype(np.uint8)
        a = [(L - n) // 2 for n in shape]
        occ = np.ascontiguousarray(o[a[0]:a[0] + shape[0], a[1]:a[1] + shape[1],
                                     a[2]:a[2] + shape[2]])
    occ[0, 0, 0] = 0
    vol = vc.upload(occ)
    vol.edt().measure()
    th = _theta(5)
    net = V.Surrogate(vc, seed=5)
    net.set_params(th)
    say("partial bricks", shape)
    _, g = net.gradients(vol)
    grow = [(0, (-n) % 8) for n in shape]
    _, g_ref = U.gradients(th.astype(np.float64), np.pad(occ, grow),
                           np.pad(vol.get(V.BUF_EDT), grow),
                           np.pad(vol.get(V.BUF_LAM2), grow), bf16=True)
    o = 0
    for name, ci, co in U.LAYERS + [("head", 16, 2)]:
        nw = (1 if name == "head" else 27) * ci * co
        rw = _rel(g[o:o + nw].astype(np.float64), g_ref[o:o + nw])
        rb = _rel(g[o + nw:o + nw + co].astype(np.float64), g_ref[o + nw:o + nw + co])
        say("partial bricks", shape, name, round(rw, 5), round(rb, 5))
        assert rw < 0.04 and rb < 0.04, (name, rw, rb)
        o += nw + co
    net.release()
    vol.release()


def test_training_lowers_loss(vc):
    """Adam on two volumes: the loss is noisy from step to step (it climbs
    for a while before it falls), so the mean of the last 10 of 60 steps is
    compared with the first loss; the last value alone depends on rounding
    (accumulation order) through the chaotic trajectory."""
    from voxel_ma_amd import surrogate
    net = V.Surrogate(vc, seed=6)
    rng = np.random.default_rng(6)
    vols = [surrogate.make_volume(vc, 64, rng) for _ in range(2)]
    losses = [net.train_step(vols, 1e-3) for _ in range(60)]
    tail = float(np.mean(losses[-10:]))
    say("train", losses[0], tail)
    assert np.all(np.isfinite(losses))
    assert tail < 0.75 * losses[0]
    for v in vols:
        v.release()
    net.release()


def test_inference_equals_training_forward(vc, small):
    """Inference runs layers 0 and 1 in one kernel, reads the decoder's
    concatenated inputs straight from the coarse level and the skip tensor,
    and evaluates the head inside the last convolution (layers 0 and 13 are
    not stored); the training forward stores every layer, materializes the
    concatenation and runs the head as its own kernel.  Both give the same
    network output, bit for bit."""
    occ, edt, lam2, vol = small
    net = V.Surrogate(vc, seed=7)
    net.set_params(_theta(7))
    net.gradients(vol)
    shape = tuple(-(-d // 8) * 8 for d in occ.shape)
    out_train = net.activation(14, shape + (2,))
    assert np.abs(out_train).max() > 0
    net.set_params(_theta(8))  # a different network in between: the output
    net.infer(vol)             # buffer must be rewritten by the next call
    assert not np.array_equal(net.activation(14, shape + (2,)), out_train)
    net.set_params(_theta(7))
    net.infer(vol)
    assert np.array_equal(net.activation(14, shape + (2,)), out_train)
    for which in (0, 13):  # not stored by an inference
        with pytest.raises(V.VcError):
            net.activation(which, shape + (16,))
    net.release()


def test_tiled_inference_equals_whole(vc):
    occ = np.zeros((80, 72, 96), np.uint8)
    occ[:, :, :] = _occ(96, 13)[:80, :72, :]
    occ[0] = occ[-1] = 0
    vol = vc.upload(occ)
    vol.edt()
    net = V.Surrogate(vc, seed=7)
    net.set_params(_theta(7))
    lam_w, rel_w = net.infer(vol, 0)
    say("tiled inference, core 32 halo", V.SURROGATE_HALO)
    lam_t, rel_t = net.infer(vol, 32)
    assert np.array_equal(lam_w, lam_t) and np.array_equal(rel_w, rel_t)
    vol.release()
    net.release()


@pytest.mark.parametrize("tau", [0.0, 0.05, 1e30])
def test_gated_measure_drives_exact_thinning(vc, oracle, tau):
    occ = _occ(48, 14)
    levels = [1.5, 3.0, 5.0]
    vol = vc.upload(occ)
    vol.edt()
    net = V.Surrogate(vc, seed=8)
    net.set_params(_theta(8))
    lam, rel = net.infer(vol)
    st = net.measure(vol, max_rel_err=tau)
    inside = occ > 0
    assert st.inside == int(inside.sum())
    assert st.accepted == int((rel[inside] <= tau).sum())
    assert st.accepted + st.fallback == st.inside
    thin = vol.thin_levels(levels)
    lab = vol.get(V.BUF_LABEL)
    # the same measure on the host: surrogate where accepted, exact otherwise
    lam2 = vol.get(V.BUF_LAM2) if st.fallback else np.zeros(occ.shape, np.uint32)
    meas = np.where(rel <= np.float32(tau), np.maximum(lam, np.float32(0)),
                    np.sqrt(lam2.astype(np.float32)))
    lvl = np.full(occ.shape, 255, np.uint8)
    for k in reversed(range(len(levels))):
        lvl[inside & (meas < np.float32(levels[k]))] = k
    lab_o, _ = oracle.thin(occ, lvl, len(levels))
    assert np.array_equal(lab, lab_o)
    # topology preserved by construction at every level
    b = oracle.betti(occ)
    for k in range(len(levels)):
        assert oracle.betti(((lab == 1) | (lab > 2 + k)).astype(np.uint8)) == b
    say("gate", tau, st.as_dict(), thin.removed[:3])
    vol.release()
    net.release()


@pytest.mark.parametrize("shape", [(2, 3, 2), (3, 5, 1), (13, 11, 23), (16, 12, 30)])
def test_gate_on_every_remainder(vc, oracle, shape):
    """The gate takes 16 and 4 voxels per access: volumes of 12, 15, 3289 and 5760
    voxels, the last voxels inside, half of the voxels accepted."""
    rng = np.random.default_rng(sum(shape))
    occ = (rng.random(shape) < 0.75).astype(np.uint8)
    occ[-1, -1] = 1
    occ[0, 0] = 0
    vol = vc.upload(occ)
    vol.edt()
    net = V.Surrogate(vc, seed=8)
    net.set_params(_theta(8))
    lam, rel = net.infer(vol)
    inside = occ > 0
    tau = float(np.median(rel[inside]))
    st = net.measure(vol, max_rel_err=tau)
    say("gate", shape, tau, st.as_dict())
    acc = rel <= np.float32(tau)
    assert st.inside == int(inside.sum()) and st.accepted == int(acc[inside].sum())
    assert st.accepted + st.fallback == st.inside and st.fallback > 0
    vol.thin_levels([0.0])
    lam2 = vol.get(V.BUF_LAM2)
    meas = np.where(acc, np.maximum(lam, np.float32(0)), np.sqrt(lam2.astype(np.float32)))
    # one level at each of the measures that occur: a voxel is a level-0 voxel
    # where its measure is below, so the levels show every value
    for t in np.unique(meas[inside])[:: max(1, inside.sum() // 40)]:
        vol.thin_levels([float(t)])
        assert np.array_equal(vol.get(V.BUF_LEVEL)[inside] == 0, meas[inside] < t), t
    vol.release()
    net.release()


def test_trained_network_gain(vc):
    """What training buys, on held-out volumes the network never saw: the
    committed weights (voxel_ma_amd/data/unet.bin, trained by
    voxel_ma_amd/surrogate.py on 4,000 volumes of 128^3) against the same
    network untrained.  The thinning with either measure is exact, so both
    skeletons keep the object's topology; training brings the measure, the
    level decisions and the skeleton towards the exact ones."""
    from voxel_ma_amd import surrogate
    rng = np.random.default_rng(2024)
    vols = [surrogate.make_volume(vc, 96, rng) for _ in range(3)]
    trained = V.Surrogate(vc, seed=1, path=surrogate.WEIGHTS)
    fresh = V.Surrogate(vc, seed=1)
    et = surrogate.evaluate(vc, trained, vols)
    eu = surrogate.evaluate(vc, fresh, vols)
    say("trained", et)
    say("untrained", eu)
    assert et["median_rel_err"] < 0.5 * eu["median_rel_err"]
    assert et["decision_agreement"] > eu["decision_agreement"]
    assert et["skeleton_iou"] > eu["skeleton_iou"]
    for v in vols:
        v.release()
    trained.release()
    fresh.release()
