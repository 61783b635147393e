"""Learned path guiding on the GPU: the FP16-MFMA network against the float64
oracle (forward outputs and loss gradients, FP16 tolerance 1e-2), the vMF
mixture probes, unbiasedness of guided renders against the unguided tracer,
and the gain of the trained network over sampling without it."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

import stats
from radiantiumplusplus_amd import _ffi as F
from radiantiumplusplus_amd import hip, scenes

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import guide_ref as G  # noqa: E402

pytestmark = pytest.mark.gpu

LO, HI = np.array([-1.0, -1.0, -1.0], np.float32), np.array([1.0, 1.0, 1.0], np.float32)


def _fp(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


def random_params(seed, out_scale=2.0):
    p = G.init_params(seed)
    rng = np.random.default_rng(seed)
    for _, bo in G.OFFS:
        p[bo:bo + 48] += rng.normal(0, 0.1, 48).astype(np.float32)
    wo, _ = G.OFFS[-1]
    p[wo:wo + 64 * 48] *= out_scale  # informative mixtures, not the near-uniform initial one
    return p


def random_feats(rng, n):
    f = np.concatenate([rng.uniform(-1, 1, (n, 3)), rng.normal(size=(n, 3)), rng.normal(size=(n, 3))], 1)
    f[:, 3:6] /= np.linalg.norm(f[:, 3:6], axis=1, keepdims=True)
    f[:, 6:9] /= np.linalg.norm(f[:, 6:9], axis=1, keepdims=True)
    return np.ascontiguousarray(f, np.float32)


def gpu_forward(p, feats):
    lib = hip.lib()
    raw = np.zeros((len(feats), 48), np.float32)
    bounds = np.concatenate([LO, HI]).astype(np.float32)
    hip.check(lib.rad_hip_guide_forward(_fp(p), _fp(bounds), _fp(feats), len(feats), _fp(raw)))
    return raw


def test_forward_matches_oracle(hip_ctx):
    rng = np.random.default_rng(0)
    p = random_params(1, out_scale=8.0)
    feats = random_feats(rng, 1000)
    raw = gpu_forward(p, feats)
    _, Z = G.forward(p, feats, LO, HI)
    ref = Z[-1]
    err = np.linalg.norm(raw - ref) / np.linalg.norm(ref)
    print(f"forward rel err {err:.2e}")
    assert err < 1e-2
    # every vertex's row, not just the aggregate
    row = np.linalg.norm(raw - ref, axis=1) / (np.linalg.norm(ref, axis=1) + 1e-3)
    assert np.quantile(row, 0.99) < 3e-2


def grad_case(p, feats, dirs, w):
    n = len(feats)
    wnorm = 1.0 / w.mean()
    recs = np.zeros(n, np.dtype([("p", "<f4", 3), ("n", "<f4", 3), ("wi", "<f4", 3), ("dir", "<f4", 3),
                                 ("thr", "<f4", 3), ("lbase", "<f4", 3), ("w", "<f4"), ("prev", "<u4")]))
    recs["p"], recs["n"], recs["wi"] = feats[:, 0:3], feats[:, 3:6], feats[:, 6:9]
    recs["dir"], recs["w"] = dirs, w
    grad = np.zeros(F.RAD_GUIDE_PARAMS, np.float32)
    loss = C.c_float()
    bounds = np.concatenate([LO, HI]).astype(np.float32)
    hip.check(hip.lib().rad_hip_guide_grad(_fp(p), _fp(bounds), recs.ctypes.data_as(C.c_void_p), n, C.c_float(wnorm),
                                           _fp(grad), C.byref(loss)))
    ref_loss, ref = G.loss_and_grad(p, feats, dirs, w.astype(np.float32), wnorm, LO, HI)
    # the same oracle on FP16-rounded weights (the weights the kernels use)
    _, ref16 = G.loss_and_grad(p.astype(np.float16).astype(np.float64), feats, dirs, w.astype(np.float32), wnorm, LO, HI)
    print(f"loss gpu {loss.value:.6f} oracle {ref_loss:.6f}")
    errs, errs16 = [], []
    for l, ((wo, bo), (nin, nout)) in enumerate(zip(G.OFFS, G.DIMS)):
        for lo_, hi_ in ((wo, bo), (bo, bo + nout)):
            e = np.linalg.norm(grad[lo_:hi_] - ref[lo_:hi_]) / (np.linalg.norm(ref[lo_:hi_]) + 1e-12)
            e16 = np.linalg.norm(grad[lo_:hi_] - ref16[lo_:hi_]) / (np.linalg.norm(ref16[lo_:hi_]) + 1e-12)
            print(f"layer {l} [{lo_}:{hi_}] rel err {e:.2e} (vs the FP16-weight oracle {e16:.2e})")
            errs.append(e)
            errs16.append(e16)
    return loss.value, ref_loss, errs, errs16


def test_gradient_matches_oracle(hip_ctx):
    """Training batches whose target directions share a common region (the
    situation guiding learns from): the FP16 gradient of every layer within
    1e-2 of the float64 oracle run on the same FP16-rounded weights, and
    within 1.5e-2 of the oracle on the FP32 weights (lobe means point from the
    vertex to a target, so the mean gradients scale with 1 / |target - vertex|
    and vertices near a target weigh the FP16 rounding of the weights more)."""
    rng = np.random.default_rng(2)
    n = 1024
    feats = random_feats(rng, n)
    axis = np.array([0.3, 0.8, -0.5]) / np.linalg.norm([0.3, 0.8, -0.5])
    dirs = axis + 0.35 * rng.normal(size=(n, 3))
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    w = rng.exponential(1.0, n)
    w[rng.random(n) < 0.2] = 0.0
    gl, rl, errs, errs16 = grad_case(random_params(3), feats, dirs, w)
    assert abs(gl - rl) <= 1e-2 * abs(rl)
    assert max(errs16) < 1e-2, errs16
    assert max(errs) < 1.5e-2, errs


def test_gradient_with_cancelling_records(hip_ctx):
    """Uniformly random target directions: the per-record gradients nearly
    cancel in the sum, so the relative error of the sum amplifies FP16
    rounding (rounding the weights alone moves the float64 oracle's own
    gradient by ~2e-2 here); bounded at 3e-2 against the oracle evaluated
    on the same FP16 weights."""
    rng = np.random.default_rng(5)
    n = 1024
    feats = random_feats(rng, n)
    dirs = rng.normal(size=(n, 3))
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    w = rng.exponential(1.0, n)
    gl, rl, _, errs16 = grad_case(random_params(4), feats, dirs, w)
    assert abs(gl - rl) <= 1e-2 * abs(rl)
    assert max(errs16) < 3e-2, errs16


@pytest.mark.parametrize("n,m", [(1, 64), (63, 65), (64, 1000), (65, 16384), (1000, 16385), (16384, 33000), (16385, 16448)])
def test_gradient_does_not_depend_on_places(hip_ctx, n, m):
    """n records, and the same records at random places among m - n of weight
    zero: other lanes, waves, tiles and blocks.  The records' gradients share a
    direction, so the two sums differ by their at most 128 roundings of 2^-24."""
    rng = np.random.default_rng(n)
    recs = np.zeros(m, np.dtype([("p", "<f4", 3), ("n", "<f4", 3), ("wi", "<f4", 3), ("dir", "<f4", 3),
                                 ("thr", "<f4", 3), ("lbase", "<f4", 3), ("w", "<f4"), ("prev", "<u4")]))
    feats = random_feats(rng, m)
    recs["p"], recs["n"], recs["wi"] = feats[:, 0:3], feats[:, 3:6], feats[:, 6:9]
    dirs = np.array([0.3, 0.8, -0.5]) + 0.2 * rng.normal(size=(m, 3))
    recs["dir"] = dirs / np.linalg.norm(dirs, axis=1, keepdims=True)
    recs["w"][:n] = rng.uniform(0.5, 1.5, n)
    p, bounds = random_params(3), np.concatenate([LO, HI]).astype(np.float32)
    out = []
    for r in (recs[:n].copy(), rng.permutation(recs)):
        grad, loss = np.zeros(F.RAD_GUIDE_PARAMS, np.float32), C.c_float()
        hip.check(hip.lib().rad_hip_guide_grad(_fp(p), _fp(bounds), r.ctypes.data_as(C.c_void_p), len(r), C.c_float(1.0),
                                               _fp(grad), C.byref(loss)))
        out.append((grad.astype(np.float64) * len(r), loss.value * len(r)))
    assert out[0][1] != 0 and abs(out[0][1] - out[1][1]) <= 1e-5 * abs(out[0][1])
    for (wo, bo), (nin, nout) in zip(G.OFFS, G.DIMS):
        for lo_, hi_ in ((wo, bo), (bo, bo + nout)):
            a, b = out[0][0][lo_:hi_], out[1][0][lo_:hi_]
            assert np.linalg.norm(a) > 0 and np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(a)


def test_mixture_probes(hip_ctx):
    rng = np.random.default_rng(4)
    raw = rng.normal(size=48).astype(np.float32)
    raw[4:40:5] = rng.uniform(-1, 3, 8)
    dirs = rng.normal(size=(4000, 3))
    dirs = (dirs / np.linalg.norm(dirs, axis=1, keepdims=True)).astype(np.float32)
    pdf = np.zeros(4000, np.float32)
    hip.check(hip.lib().rad_hip_guide_pdf(_fp(raw), _fp(dirs), 4000, _fp(pdf)))
    assert np.allclose(pdf, G.pdf(raw, dirs), rtol=1e-4, atol=1e-7)
    n = 200000
    xi = rng.random((n, 3)).astype(np.float32)
    out = np.zeros((n, 4), np.float32)
    hip.check(hip.lib().rad_hip_guide_sample(_fp(raw), _fp(xi), n, _fp(out)))
    d = out[:, :3].astype(np.float64)
    assert np.allclose(np.linalg.norm(d, axis=1), 1.0, atol=1e-5)
    assert np.allclose(out[:, 3], G.pdf(raw, d), rtol=1e-3, atol=1e-6)
    # the samples follow the density: E[d] and E[d_y^2] against quadrature of the pdf
    t = (np.arange(400) + 0.5) * np.pi / 400
    f = (np.arange(800) + 0.5) * 2 * np.pi / 800
    T, P = np.meshgrid(t, f, indexing="ij")
    q = np.stack([np.sin(T) * np.cos(P), np.cos(T), np.sin(T) * np.sin(P)], -1).reshape(-1, 3)
    dw = (np.sin(T) * (np.pi / 400) * (2 * np.pi / 800)).reshape(-1)
    pq = G.pdf(raw, q) * dw
    for k, fn in enumerate([lambda v: v[:, 0], lambda v: v[:, 1], lambda v: v[:, 2], lambda v: v[:, 1] ** 2]):
        expect = (fn(q) * pq).sum()
        vals = fn(d)
        se = vals.std() / np.sqrt(n)
        assert abs(vals.mean() - expect) < 5 * se + 1e-4, (k, vals.mean(), expect, se)


def small_room(width=48, height=27):
    b = scenes.guiding_room(width=width, height=height, spp=256)
    return b


def render(ctx, scene, b, spp, seed, guiding=0, flags=0):
    rd = b.render_desc(spp=spp, seed=seed, flags=flags | F.RAD_RENDER_WANT_SUMSQ)
    rd.guiding = guiding
    return scene.render(rd, want_sumsq=True)


def test_guided_render_is_unbiased(hip_ctx):
    """Guided (online-trained) and unguided renders of the door-gap room
    converge to the same image: per-tile z-test at 4 sigma."""
    b = small_room()
    s = hip.Scene.from_builder(hip_ctx, b)
    fb_p, sq_p, _ = render(hip_ctx, s, b, 4096, seed=1, guiding=0)
    fb_g, sq_g, st = render(hip_ctx, s, b, 4096, seed=2, guiding=1)
    print(f"guide steps {st.guide_steps} records {st.guide_records} loss {st.guide_loss:.4f} alpha {st.guide_alpha}")
    assert st.guide_steps > 0 and st.guide_alpha > 0
    assert np.isfinite(fb_g).all()
    z, rel = stats.compare(fb_g, sq_g, 4096, fb_p, sq_p, 4096, tile=8)
    print(f"max |z| {np.abs(z).max():.2f}  relMSE {rel:.2e}")
    assert np.abs(z).max() < 4.0
    assert rel < 2e-3


def test_guided_queues_are_a_permutation(hip_ctx):
    """With guiding or training records on, classify puts each material's
    guided vertices at the back of its queue and the rest at the front: the
    device tally finds every extension-queue slot exactly once, each guided
    entry where the guided-vertex test holds and no unguided entry where it
    does, through training passes (records, no guide) and guided passes.
    The check leaves a fixed-weight guided image unchanged."""
    b = small_room()
    s = hip.Scene.from_builder(hip_ctx, b)
    rd = b.render_desc(spp=1024, seed=3, flags=F.RAD_RENDER_CHECK_QUEUES)
    rd.guiding = 1
    _, _, st = s.render(rd)
    print(f"guide steps {st.guide_steps} checked {st.queue_checked} errors {st.queue_errors}")
    assert st.guide_steps > 0 and st.guide_alpha > 0
    assert st.queue_errors == 0 and st.queue_checked == st.segments + st.suspended > 0
    ref, _, _ = render(hip_ctx, s, b, 64, seed=4, guiding=2)
    img, _, st2 = render(hip_ctx, s, b, 64, seed=4, guiding=2, flags=F.RAD_RENDER_CHECK_QUEUES)
    assert st2.queue_errors == 0 and st2.queue_checked == st2.segments + st2.suspended > 0
    assert np.array_equal(img, ref)


def test_unsorted_guided_render_matches_sorted(hip_ctx):
    """The single-kernel guided path (guide queue of extend-queue positions,
    outputs in rows by position, one shading kernel for every vertex)
    converges to the material-sorted guided path's image: per-tile z-test at
    4 sigma, fixed trained weights, different seeds."""
    b = small_room()
    s = hip.Scene.from_builder(hip_ctx, b)
    rd = b.render_desc(spp=256, seed=3)
    rd.guiding = 1
    _, _, st = s.render(rd)
    assert st.guide_steps > 0
    fa, qa, sa = render(hip_ctx, s, b, 1024, seed=4, guiding=2)
    fu, qu, su = render(hip_ctx, s, b, 1024, seed=5, guiding=2, flags=F.RAD_RENDER_UNSORTED)
    assert sa.guide_alpha > 0 and su.guide_alpha > 0
    z, rel = stats.compare(fa, qa, 1024, fu, qu, 1024, tile=8)
    print(f"max |z| {np.abs(z).max():.2f}  relMSE {rel:.2e}")
    assert np.abs(z).max() < 4.0
    assert rel < 2e-3


def test_trained_guide_reduces_error(hip_ctx):
    """At equal spp the trained guide's error against a converged unguided
    reference is well below that of BSDF sampling alone (quirks off, so the
    GGX boxes are guided too).  The guide lives in scene space, so it is
    trained on a 640x360 render of the room (about 6M training records) and
    evaluated on a 64x36 one; measured ratio about 0.5."""
    b = small_room(64, 36)
    fl = F.RAD_RENDER_FIX_QUIRKS
    s = hip.Scene.from_builder(hip_ctx, b)
    ref, _, _ = render(hip_ctx, s, b, 16384, seed=10, flags=fl)
    # train once (guiding = 1), then compare fixed-weight guiding (2) with plain sampling at 64 spp
    rd = b.render_desc(spp=256, seed=11, flags=fl)
    rd.guiding, rd.width, rd.height = 1, 640, 360
    _, _, st = s.render(rd)
    assert st.guide_steps > 0 and st.guide_records > 1000000
    errs_p, errs_g = [], []
    for k in range(4):
        fp, _, _ = render(hip_ctx, s, b, 64, seed=100 + k, guiding=0, flags=fl)
        fg, _, _ = render(hip_ctx, s, b, 64, seed=200 + k, guiding=2, flags=fl)
        errs_p.append(np.mean((fp - ref) ** 2 / (ref ** 2 + 1e-2)))
        errs_g.append(np.mean((fg - ref) ** 2 / (ref ** 2 + 1e-2)))
    mp, mg = np.mean(errs_p), np.mean(errs_g)
    print(f"relMSE plain {mp:.4e} guided {mg:.4e} ratio {mg / mp:.3f}")
    assert mg < 0.75 * mp
