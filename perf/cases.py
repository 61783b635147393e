"""Workloads that a user of the renderer has it do, for timing and comparing builds.

Each case goes through the public entry points: ray queries on a resident
scene (`Scene.closest`, `rad_hip_intersect_*_device`), tree builds
(`Scene.build_bvh`), renders with the `path` and `vol_path` integrators
(`Scene.render`), the guide's training gradient (`rad_hip_guide_grad`) and
the render server (`serve.Server`).  Scenes are the package's own generators.

`run` returns whole images, hit records and gradients.  Images are a function
of the scene and the seed alone, whatever order the samples are traced in.
"""
import ctypes as C
import math

import numpy as np
import torch

from radiantiumplusplus_amd import _ffi as F
from radiantiumplusplus_amd import hip, scenes, serve

_ctx = None
_lib = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = hip.Context(0)
    return _ctx


def _native():
    """The C ABI with the argument types of the entry points that hip.py leaves to callers."""
    global _lib
    if _lib is None:
        _lib = hip.lib()
    return _lib


# --------------------------------------------------------------------------- cases
def listed():
    return [
        # An editor or tool asks what lies under a few cursor positions or probe rays: latency of one small call
        # on host arrays.
        {"name": "probe_rays_host", "kind": "closest_host", "spheres": 64, "rays": 1500},
        # Visibility and distance queries of a program that keeps its rays on the GPU (light baking, a custom
        # integrator): incoherent rays over a terrain, closest hit and occlusion; an odd count.
        {"name": "closest_rays_device", "kind": "closest", "grid": 512, "spheres": 96, "rays": 3000001},
        {"name": "occlusion_rays_device", "kind": "any", "grid": 512, "spheres": 96, "rays": 4000000},
        # The scene changed: the tree is built again and queried.
        {"name": "tree_build_terrain", "kind": "build", "grid": 1024, "spheres": 256, "rays": 65536},
        # A thumbnail: the smallest render, where launches and host work count.
        {"name": "render_thumbnail", "kind": "render", "scene": "balls", "spheres": 64, "width": 64, "height": 48,
         "spp": 4, "guiding": 0, "slots": 0},
        # The plain path tracer at its default size (diffuse spheres, one area light).
        {"name": "render_balls", "kind": "render", "scene": "balls", "spheres": 64, "width": 512, "height": 512,
         "spp": 16, "guiding": 0, "slots": 0},
        # Every material and texture type at an odd size: the shading kernels that the other scenes leave out.
        {"name": "render_materials", "kind": "render", "scene": "materials", "width": 637, "height": 397, "spp": 32,
         "guiding": 0, "slots": 0},
        # The headline frame: 8.9 M triangles, 1080p, 64 samples, the launch configuration the autotuner finds.
        {"name": "render_terrain_1080p", "kind": "render", "scene": "terrain", "grid": 2048, "spheres": 256,
         "width": 1920, "height": 1080, "spp": 64, "guiding": 0, "slots": 67108864},
        # Heterogeneous medium, vol_path, at its default size.
        {"name": "render_volume", "kind": "render", "scene": "volume", "grid": 256, "width": 1024, "height": 1024,
         "spp": 64, "guiding": 0, "slots": 0},
        # Difficult indirect light with a guide in hand: network inference inside the tracer.
        {"name": "render_room_guided", "kind": "render", "scene": "room", "width": 1280, "height": 720, "spp": 32,
         "guiding": 2, "slots": 0},
        # One gradient of the guide's loss: the training direction of the network.
        {"name": "guide_gradient", "kind": "grad", "records": 32768},
        # A render server with small and ordinary requests of three scenes in flight together.
        {"name": "serve_mixed", "kind": "serve", "requests": 8, "grid": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest_host", "closest", "any", "build", "render", "render", "render", "render", "grad", "serve"])
    if kind == "closest_host":
        return {"kind": kind, "spheres": rng.randint(8, 200), "rays": _log(rng, 1, 200000)}
    if kind in ("closest", "any"):
        return {"kind": kind, "grid": _log(rng, 32, 1024), "spheres": rng.randint(3, 256), "rays": _log(rng, 1000, 8000000)}
    if kind == "build":
        return {"kind": kind, "grid": _log(rng, 16, 1400), "spheres": rng.randint(3, 256), "rays": _log(rng, 1000, 100000)}
    if kind == "grad":
        return {"kind": kind, "records": _log(rng, 500, 100000)}
    if kind == "serve":
        return {"kind": kind, "requests": rng.randint(2, 12), "grid": _log(rng, 64, 512)}
    scene = rng.choice(["balls", "materials", "terrain", "volume", "room"])
    w = _log(rng, 33, 1920)
    h = max(17, int(w * rng.uniform(0.5, 1.0)))
    case = {"kind": kind, "scene": scene, "width": w, "height": h,
            "spp": max(1, min(64, _log(rng, 1, 64), 40000000 // (w * h))), "guiding": 0, "slots": 0}
    if scene == "balls":
        case["spheres"] = rng.randint(8, 200)
    if scene == "terrain":
        case["grid"] = _log(rng, 64, 1024)
        case["spheres"] = rng.randint(3, 256)
        case["slots"] = rng.choice([0, 16777216])
    if scene == "volume":
        case["grid"] = _log(rng, 16, 200)
    if scene == "room":
        case["guiding"] = rng.choice([0, 2])
    return case


# --------------------------------------------------------------------------- scenes
def _materials(seed, width, height, spp):
    """Every BSDF type the specialised kernels leave to the generic one, textured parameters, a mesh with
    uvs, and area, point and projection lights (the scenes of the BSDF and texture tests, together)."""
    rng = np.random.default_rng(seed)
    b = scenes.SceneBuilder()
    img = rng.uniform(0.1, 0.9, (64, 64, 3)).astype(np.float32)
    img[::8] *= 0.3
    mono = rng.uniform(0.05, 0.5, (16, 16)).astype(np.float32)
    cb = b.chessboard(color_a=(0.8, 0.2, 0.2), color_b=b.bitmap(img, filter="anisotropic"),
                      to_uv=scenes.trs(scale=(4, 4, 1)), remap=True)
    b.rectangle(to_world=scenes.trs(axis=(1, 0, 0), angle=-90, scale=(6, 6, 6)),
                bsdf=b.diffuse(b.bitmap(img, filter="trilinear", wrap="repeat")))
    mats = [b.plastic(diffuse=(0.7, 0.2, 0.2)), b.rough_plastic(alpha=0.3, diffuse=(0.2, 0.6, 0.3)),
            b.perfect_mirror(reflectance=(0.9, 0.9, 0.8), eta=(0.2, 0.9, 1.1), k=(3.9, 2.4, 2.1)),
            b.perfect_glass(int_ior=1.5, ext_ior=1.0), b.mask(b.diffuse((0.3, 0.3, 0.8)), opacity=0.5),
            b.rough_metal(alpha=b.bitmap(mono, filter="nearest"), reflectance=cb),
            b.rough_glass(alpha=0.1, int_ior=1.5, ext_ior=1.0), b.disney(base_color=(0.6, 0.5, 0.2), roughness=0.4, metallic=0.7),
            b.plastic(diffuse=b.bitmap(img, filter="bilinear")), b.rough_metal(alpha=0.2)]
    for i, m in enumerate(mats):
        b.sphere(center=(-3.4 + 1.7 * (i % 5), 0.7, -0.6 + 2.2 * (i // 5) + rng.uniform(-0.2, 0.2)), radius=0.7, bsdf=m)
    p, _, uv, idx = scenes.create_sphere(0.6, 24)
    b.mesh(p, idx, uvs=uv, to_world=scenes.trs(translate=(0.2, 0.6, -2.2)),
           bsdf=b.disney(base_color=b.bitmap(img, filter="nearest"), roughness=0.4, metallic=b.bitmap(mono)))
    b.rectangle(to_world=scenes.trs(translate=(0, 1.5, 3.5), scale=(3.5, 1.5, 1)), bsdf=b.two_side(b.diffuse(0.7)))
    light = b.rectangle(to_world=scenes.trs(translate=(0, 5, -1), axis=(1, 0, 0), angle=90, scale=(1, 1, 1)))
    b.area_light(light, 6.0)
    b.point_light((2.5, 3.0, -2.0), (12.0, 10.0, 8.0))
    tw = np.array([[1, 0, 0, -2.0], [0, 0, -1, 4.0], [0, 1, 0, -1.0], [0, 0, 0, 1]], np.float32)
    b.projection_light(tw, irradiance=(0.8, 0.9, 1.0), scale=2.0, fov=35.0)
    b.set_camera(width, height, 55, origin=(0, 3, -8), target=(0, 0.8, 0), far=1000)
    b.set_render("path", spp=spp, max_depth=10, rr_depth=3, seed=seed)
    return b


def _builder(case, seed):
    w, h, spp = case.get("width", 64), case.get("height", 64), case.get("spp", 1)
    which = case.get("scene") or ("balls" if case["kind"] == "closest_host" else "terrain")
    if which == "balls":
        return scenes.many_balls(seed=seed, width=w, height=h, spp=spp, n_spheres=case["spheres"])
    if which == "materials":
        return _materials(seed, w, h, spp)
    if which == "terrain":
        return scenes.large_mesh(seed=seed, width=w, height=h, spp=spp, grid=case["grid"], n_spheres=case["spheres"])
    if which == "volume":
        return scenes.volume_box(seed=seed, width=w, height=h, spp=spp, res=case["grid"])
    return scenes.guiding_room(seed=seed, width=w, height=h, spp=spp)


def _guide_weights(seed):
    """Network weights of the size that training arrives at: He-uniform layers, outputs of order one."""
    rng = np.random.default_rng(seed)
    p = np.zeros(F.RAD_GUIDE_PARAMS, np.float32)
    o = 0
    for nin, nout in _DIMS:
        lim = math.sqrt(6.0 / nin)
        p[o:o + nin * nout] = rng.uniform(-lim, lim, nin * nout)
        o += nin * nout
        p[o:o + nout] = rng.uniform(-0.1, 0.1, nout)
        o += nout
    return p


_DIMS = [(80, 64), (64, 64), (64, 64), (64, 64), (64, 48)]
_RECORD = np.dtype([("p", "<f4", 3), ("n", "<f4", 3), ("wi", "<f4", 3), ("dir", "<f4", 3), ("thr", "<f4", 3),
                    ("lbase", "<f4", 3), ("w", "<f4"), ("prev", "<u4")])
_LO, _HI = (-3.0, 0.0, -3.0), (9.5, 3.0, 3.0)


def _terrain_rays(seed, n):
    """n x 8 device floats: origins over the terrain, half cosine-like directions (bounces), half any direction
    (a third of them near-grazing), a fifth with short segments."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    u = lambda *s: torch.rand(*s, generator=g, device="cuda")  # noqa: E731
    r = torch.empty(n, 8, device="cuda")
    r[:, 0:3] = u(n, 3) * torch.tensor([40.0, 5.0, 40.0], device="cuda") + torch.tensor([-20.0, -1.0, -20.0], device="cuda")
    d = torch.randn(n, 3, generator=g, device="cuda")
    up = u(n) < 0.5
    d[:, 1] = torch.where(up, d[:, 1].abs() + 0.2, torch.where(u(n) < 0.33, d[:, 1] * 0.05, d[:, 1]))
    r[:, 4:7] = d / d.norm(dim=1, keepdim=True).clamp_min(1e-6)
    r[:, 3] = 0.0
    r[:, 7] = torch.where(u(n) < 0.2, u(n) * 5.0 + 0.1, torch.full((n,), 1.0e3, device="cuda"))
    return r


def _ball_rays(seed, n):
    rng = np.random.default_rng(seed)
    rays = np.zeros(n, hip.RAY_DTYPE)
    rays["o"] = rng.uniform([-6, 0.1, -6], [6, 6, 6], (n, 3))
    d = rng.normal(size=(n, 3))
    rays["d"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmax"] = 100.0
    return rays


def _records(seed, n):
    """Vertices of the room with sampled directions and weights as paths record them (most small, a few large)."""
    rng = np.random.default_rng(seed)
    r = np.zeros(n, _RECORD)

    def unit(k):
        v = rng.normal(size=(k, 3))
        return v / np.linalg.norm(v, axis=1, keepdims=True)

    r["p"] = rng.uniform([-3, 0, -3], [3, 3, 3], (n, 3))
    r["n"], r["wi"] = unit(n), unit(n)
    to = np.array([-3.0, 1.5, 0.0]) + rng.normal(size=(n, 3)) * 0.4 - r["p"]
    r["dir"] = np.where((rng.random(n) < 0.6)[:, None], to / np.linalg.norm(to, axis=1, keepdims=True), unit(n))
    r["w"] = rng.exponential(1.0, n) ** 2
    r["prev"] = 0xFFFFFFFF
    return r


# --------------------------------------------------------------------------- prepare / run
def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    s = {"kind": kind}
    if kind == "grad":
        s["params"], s["recs"] = _guide_weights(seed), _records(seed, case["records"])
        s["bounds"] = np.array(_LO + _HI, np.float32)
        s["wnorm"] = 1.0 / float(s["recs"]["w"].mean())
        return s
    if kind == "serve":
        rng = np.random.default_rng(seed)
        s["builders"] = {"balls": scenes.many_balls(seed=seed, n_spheres=64),
                         "terrain": scenes.large_mesh(seed=seed, grid=case["grid"], n_spheres=24),
                         "volume": scenes.volume_box(seed=seed, res=64)}
        s["scenes"] = {k: hip.Scene.from_builder(ctx, b) for k, b in s["builders"].items()}
        s["server"] = serve.Server(ctx, hbm_budget=32 << 30, max_inflight=8)
        names = list(s["builders"])
        s["requests"] = []
        for i in range(case["requests"]):
            w, h = [(256, 256), (512, 512), (1024, 1024), (400, 225)][i % 4]
            d = s["builders"][names[i % 3]].render_desc(spp=[4, 16, 8][(i // 2) % 3], seed=int(rng.integers(1 << 30)),
                                                        request_id=i + 1)
            d.width, d.height = w, h
            s["requests"].append((names[i % 3], d))
        return s
    b = _builder(case, seed)
    s["scene"] = hip.Scene.from_builder(ctx, b)
    if kind == "closest_host":
        s["rays"] = _ball_rays(seed, case["rays"])
    elif kind == "render":
        s["desc"] = b.render_desc(seed=seed, path_slots=case["slots"], guiding=case["guiding"])
        if case["guiding"]:
            s["scene"].set_guide_params(_guide_weights(seed))
    else:
        n = case["rays"]
        s["rays"] = _terrain_rays(seed, n)
        s["hits"] = torch.zeros(n, 5, dtype=torch.int32, device="cuda")
        s["occluded"] = torch.zeros(n, dtype=torch.uint8, device="cuda")
    return s


def _hits(h):
    f = h.view(torch.float32)
    return {"t": f[:, 0], "uv": f[:, 1:3], "ids": h[:, 3:5]}


def run(s):
    kind = s["kind"]
    if kind == "closest_host":
        h = s["scene"].closest(s["rays"])
        return {"t": h["t"], "uv": np.stack([h["u"], h["v"]], 1), "ids": np.stack([h["prim"], h["geom"]], 1).view(np.int32)}
    if kind == "render":
        return s["scene"].render(s["desc"])[0]
    if kind == "grad":
        grad, loss = np.zeros(F.RAD_GUIDE_PARAMS, np.float32), C.c_float()
        hip.check(_native().rad_hip_guide_grad(s["params"].ctypes.data, s["bounds"].ctypes.data, s["recs"].ctypes.data,
                                               len(s["recs"]), s["wnorm"], grad.ctypes.data, C.byref(loss)))
        return {"grad": grad, "loss": float(loss.value)}
    if kind == "serve":
        ids = [s["server"].submit(s["scenes"][name], d) for name, d in s["requests"]]
        return [s["server"].wait(i).image for i in ids]
    rays, n, stream = s["rays"], s["rays"].shape[0], torch.cuda.current_stream().cuda_stream
    if kind == "any":
        hip.check(_native().rad_hip_intersect_any_device(s["scene"].h, rays.data_ptr(), n, s["occluded"].data_ptr(), stream))
        return s["occluded"]
    if kind == "build":
        s["scene"].build_bvh()
    hip.check(_native().rad_hip_intersect_closest_device(s["scene"].h, rays.data_ptr(), n, s["hits"].data_ptr(), stream))
    return _hits(s["hits"])


# --------------------------------------------------------------------------- work, tolerance, exact
def _triangles(case):
    which = case.get("scene") or ("balls" if case["kind"] == "closest_host" else "terrain")
    if which == "balls":
        return 1024 * case["spheres"] + 2
    if which == "terrain":
        return 2 * (case["grid"] - 1) ** 2 + 2116 * case["spheres"] + 1
    return {"materials": 600, "volume": 19, "room": 400}[which]


def _ray_ops(prims):
    """Floating operations that a ray through a 4-wide tree cannot do without: one descent to a leaf (four boxes of
    13 operations a level) and two triangle tests."""
    return 52.0 * max(1.0, math.log(max(prims, 4) / 4.0, 4.0)) + 2 * 60.0


def _render_work(prims, w, h, spp, scene, guiding):
    n = float(w * h * spp)
    # rays a sample needs on average (closest hit and occlusion together), as these scenes' renders count them
    rays = {"balls": 3.0, "materials": 5.0, "terrain": 3.2, "volume": 6.0, "room": 12.0}[scene]
    flops = n * rays * (_ray_ops(prims) + 200.0)
    if guiding:
        flops += n * 3 * 2.0 * sum(a * b for a, b in _DIMS)
    return {"bytes": 12.0 * w * h + 48.0 * prims, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "grad":
        n = float(case["records"])
        return {"bytes": 80.0 * n + 8.0 * F.RAD_GUIDE_PARAMS, "flops": 6.0 * n * sum(a * b for a, b in _DIMS)}
    if kind == "serve":
        out = {"bytes": 0.0, "flops": 0.0}
        for i in range(case["requests"]):
            w, h = [(256, 256), (512, 512), (1024, 1024), (400, 225)][i % 4]
            scene = ["balls", "terrain", "volume"][i % 3]
            prims = {"balls": 65538, "terrain": 2 * (case["grid"] - 1) ** 2 + 2116 * 24, "volume": 19}[scene]
            k = _render_work(prims, w, h, [4, 16, 8][(i // 2) % 3], scene, 0)
            out = {m: out[m] + k[m] for m in out}
        return out
    prims = _triangles(case)
    if kind == "render":
        return _render_work(prims, case["width"], case["height"], case["spp"], case["scene"], case["guiding"])
    n = float(case["rays"])
    out = {"bytes": n * (33.0 if kind == "any" else 52.0), "flops": n * _ray_ops(prims)}
    if kind == "build":  # primitive boxes and records in; 64-byte nodes (one per three primitives) and records out
        out["bytes"] += prims * (24.0 + 48.0 + 64.0 / 3 + 48.0)
    return out


def tolerance(case):
    """Measured by comparing the build with one whose floating contraction is off (every product and sum of the
    shading code rounds differently; a rounding that flips one decision of a path replaces that sample): four times
    the differences seen.  Hits: another builder's tree over the same primitives gave the same hits bit for bit;
    a tie between two primitives may go either way."""
    kind = case["kind"]
    if kind == "any":
        return "exact"
    if kind == "grad":  # seen: 1.3e-6, largest 1.5e-5
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "serve":  # seen: 7e-5, largest 0.1
        return {"rel": 1e-3, "max": 0.5}
    if kind == "render":
        if case["guiding"]:  # seen: 9.5e-3, largest 1.8 (FP16 network outputs steer whole paths)
            return {"rel": 0.03, "max": 0.99}
        if case["scene"] == "volume":  # seen: 1.4e-5 on 67 M samples, largest 0.011
            return {"rel": 1e-3, "max": 0.5}
        return {"rel": 3e-3, "max": 0.95}  # seen: 7.2e-4, largest 0.23
    return {"rel": 1e-3, "max": 0.99, "differ": 1e-5}


def exact(case, seed):
    if case["kind"] == "grad":
        return _exact_grad(case, seed)
    if case["kind"] == "closest_host" and case["rays"] * case["spheres"] <= 400000:
        return _exact_hits(case, seed)
    return None


def _exact_grad(case, seed):
    """The mean negative log likelihood of the recorded directions under the network's 8-lobe von Mises-Fisher
    mixture, and its gradient by automatic differentiation, in 64 bits."""
    dev = torch.device("cuda")
    d64 = lambda a: torch.tensor(np.asarray(a, np.float64), device=dev)  # noqa: E731
    recs = _records(seed, case["records"])
    p = d64(_guide_weights(seed)).requires_grad_()
    lo, hi = d64(_LO), d64(_HI)
    pos, nrm, wi, dirs, w = (d64(recs[k]) for k in ("p", "n", "wi", "dir", "w"))
    wn = (w * float(np.float32(1.0 / float(recs["w"].mean())))).clamp(max=64.0)
    s = [((pos - lo) / (hi - lo)).clamp(0, 1)]
    for v in (nrm, wi):
        s.append(torch.stack([(0.5 * (v[:, 1] + 1)).clamp(0, 1), torch.atan2(v[:, 2], v[:, 0]) / (2 * math.pi) + 0.5], 1))
    s = torch.cat(s, 1)
    x = torch.cat([(1 - (s[:, k:k + 1] * n - (torch.arange(n, device=dev) + 0.5)).abs()).clamp(min=0)
                   for k, n in enumerate([16, 16, 16, 8, 8, 8, 8])], 1)
    o = 0
    for i, (nin, nout) in enumerate(_DIMS):
        x = x @ p[o:o + nin * nout].reshape(nout, nin).T + p[o + nin * nout:o + nin * nout + nout]
        o += nin * nout + nout
        if i < 4:
            x = x.relu()
    raw = x[:, :40].reshape(-1, 8, 5)
    mu = 0.5 * (lo + hi) + 0.5 * (hi - lo) * raw[:, :, 1:4] - pos[:, None, :]
    mu = mu / mu.norm(dim=2, keepdim=True)
    kappa = raw[:, :, 4].clamp(-3, 6).exp()
    lv = kappa.log() - math.log(2 * math.pi) - torch.log1p(-torch.exp(-2 * kappa)) + kappa * ((mu * dirs[:, None, :]).sum(2) - 1)
    loss = -(wn * torch.logsumexp(torch.log_softmax(raw[:, :, 0], 1) + lv, 1)).mean()
    loss.backward()
    return {"grad": p.grad, "loss": float(loss.detach())}


def _exact_hits(case, seed):
    """Closest hits by testing every triangle and rectangle, in 64 bits (ids have no 64-bit value)."""
    dev = torch.device("cuda")
    d64 = lambda a: torch.tensor(np.asarray(a, np.float64), device=dev)  # noqa: E731
    b = _builder(case, seed)
    rays = _ball_rays(seed, case["rays"])
    o, d = d64(rays["o"]), d64(rays["d"])
    t = torch.full((len(rays),), 100.0, dtype=torch.float64, device=dev)
    uv = torch.zeros(len(rays), 2, dtype=torch.float64, device=dev)

    def closer(tt, u, v):
        nonlocal t, uv
        best, k = tt.min(1)
        hit = best < t
        t = torch.where(hit, best, t)
        uv = torch.where(hit[:, None], torch.stack([u.gather(1, k[:, None])[:, 0], v.gather(1, k[:, None])[:, 0]], 1), uv)

    for sh in b.shapes:
        m = d64(sh.to_world)
        if sh.kind == "mesh":
            pos, _, _, idx = sh.mesh
            v = (d64(pos) @ m[:3, :3].T + m[:3, 3])[torch.tensor(idx.reshape(-1, 3).astype(np.int64), device=dev)]
            v0, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
            n = torch.linalg.cross(e1, e2)
            den = -(d @ n.T)
            to = o[:, None, :] - v0[None]
            q = torch.linalg.cross(to, d[:, None, :].expand_as(to))
            tt, u, w = (to * n).sum(2) / den, (q * e2).sum(2) / den, -(q * e1).sum(2) / den
            ok = (den != 0) & (u >= 0) & (w >= 0) & (u + w <= 1) & (tt > 0)
        else:
            inv = torch.linalg.inv(m)
            lo, ld = o @ inv[:3, :3].T + inv[:3, 3], d @ inv[:3, :3].T
            tt = (-lo[:, 2] / ld[:, 2])[:, None]
            at = lo + ld * tt
            u, w = at[:, 0:1], at[:, 1:2]
            ok = (tt > 0) & (u.abs() <= 1) & (w.abs() <= 1)
        closer(torch.where(ok, tt, torch.full_like(tt, math.inf)), u, w)
    return {"t": t, "uv": uv, "ids": None}
