"""The device BVH builder (Morton-ordered binned SAH + 4-wide collapse):
closest / any hit parity with the oracle's brute force, structural
invariants (every primitive referenced once, child boxes inside the parent,
leaf boxes around their primitives), SAH cost within a band of the host
binned-SAH builder, and renders that match the host-built tree."""
import numpy as np
import pytest

import _oracle as O
from _trees import mesh_scene, shrinking_sequence
from radiantiumplusplus_amd import _ffi as F
from radiantiumplusplus_amd import hip, scenes
from test_gpu_intersect import check_parity, ray_batch

pytestmark = pytest.mark.gpu


def terrain_scene(grid=256, spheres=32, seed=5):
    rng = np.random.default_rng(seed)
    b = scenes.SceneBuilder()
    p, n, uv, idx = scenes.create_grid(20, 20, grid, grid)
    h = scenes.fbm_heightfield(grid, grid, 6, 2.0, seed)
    p = p.copy()
    p[:, 1] += h.reshape(-1)
    b.mesh(p, idx, None, uv, bsdf=b.diffuse(0.5))
    for _ in range(spheres):
        c = rng.uniform([-8, 1, -8], [8, 3, 8])
        sp, sn, su, si = scenes.create_sphere(rng.uniform(0.2, 0.8), 16)
        b.mesh(sp, si, sn, su, to_world=scenes.trs(translate=c), bsdf=b.diffuse(0.6))
    b.sphere(center=(0, 4, 0), radius=0.5, bsdf=b.diffuse(0.5))
    b.rectangle(to_world=scenes.trs(translate=(0, 6, 0), axis=(1, 0, 0), angle=90, scale=(2, 2, 2)))
    b.area_light(len(b.shapes) - 1, 5.0)
    b.set_camera(32, 32, 45, origin=(0, 8, -18), target=(0, 0, 0), far=1000)
    b.set_render("path", spp=4, max_depth=6)
    return b


@pytest.mark.parametrize("seed", [0, 1])
def test_device_bvh_closest_hit_matches_brute_force(hip_ctx, seed):
    b = scenes.many_balls(seed=seed, n_spheres=64, slices=32, width=16, height=16)
    o = O.OracleScene(b)
    g = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_DEVICE)
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, 20000, seed)
    ties = check_parity(o, rays, g.closest(rays), o.closest(rays, brute=True))
    assert ties <= 10


def test_device_bvh_terrain_parity_and_structure(hip_ctx):
    b = terrain_scene()
    o = O.OracleScene(b)
    g = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_DEVICE)
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, 5000, 7)
    ties = check_parity(o, rays, g.closest(rays), o.closest(rays, brute=True))
    assert ties <= 10
    occ = g.occluded(rays)
    assert np.array_equal(occ.astype(bool), o.occluded(rays, brute=True).astype(bool))
    r = g.bvh_check()
    assert r.builder == F.RAD_BVH_DEVICE
    assert r.structure_errors == 0 and r.unreferenced_or_repeated == 0
    assert r.child_box_violations == 0 and r.leaf_box_violations == 0
    assert r.quantized_box_violations == 0
    assert r.max_leaf <= 4
    h = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_HOST).bvh_check()
    assert h.structure_errors == 0 and h.unreferenced_or_repeated == 0 and h.quantized_box_violations == 0
    print(f"SAH device {r.sah_cost:.2f} host {h.sah_cost:.2f} ratio {r.sah_cost / h.sah_cost:.3f}; "
          f"depth {r.depth} / {h.depth}; nodes {r.node_count} / {h.node_count}")
    assert r.sah_cost <= 1.10 * h.sah_cost


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 1000])
def test_device_bvh_small_counts(hip_ctx, n):
    """Root-leaf and tiny trees around the leaf size and the exact-sweep size."""
    rng = np.random.default_rng(n)
    b = scenes.SceneBuilder()
    for _ in range(n):
        b.sphere(center=tuple(rng.uniform(-5, 5, 3)), radius=float(rng.uniform(0.1, 0.4)), bsdf=b.diffuse(0.5))
    b.skybox(1.0)
    b.set_camera(8, 8, 45, origin=(0, 0, -20), target=(0, 0, 0), far=100)
    o = O.OracleScene(b)
    g = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_DEVICE)
    r = g.bvh_check()
    assert r.structure_errors == 0 and r.unreferenced_or_repeated == 0 and r.leaf_box_violations == 0
    assert r.quantized_box_violations == 0
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, 4000, n)
    check_parity(o, rays, g.closest(rays), o.closest(rays, brute=True))


def test_device_bvh_render_matches_host_bvh(hip_ctx):
    b = scenes.many_balls(seed=2, width=48, height=48, spp=16, n_spheres=32)
    gd = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_DEVICE)
    gh = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_HOST)
    a = gd.render(b.render_desc(spp=64, seed=3))[0]
    c = gh.render(b.render_desc(spp=64, seed=3))[0]
    # same closest hits up to distance ties: identical samples almost everywhere
    assert np.mean(a != c) < 1e-3


def nested_clumps(levels, seed=0):
    """Clumps of six small triangles at geometrically shrinking scales: at
    each scale three clumps sit around a smaller copy of the rest, so every
    4-wide level can hold three inner siblings and the traversal stack need
    grows with the number of levels."""
    rng = np.random.default_rng(seed)
    pts, centres = [], []
    for i in range(levels):
        s = 0.45 ** i
        for axis in range(3):
            c = np.zeros(3)
            c[axis] = 0.8 * s
            centres.append(c)
            for _ in range(6):
                p0 = c + rng.normal(0, 0.04 * s, 3)
                pts += [p0, p0 + rng.normal(0, 0.03 * s, 3), p0 + rng.normal(0, 0.03 * s, 3)]
    b = scenes.SceneBuilder()
    b.mesh(np.array(pts, np.float32), np.arange(len(pts), dtype=np.uint32), bsdf=b.diffuse(0.5))
    b.skybox(1.0)
    b.set_camera(8, 8, 45, origin=(0, 0, -5), target=(0, 0, 0), far=100)
    return b, np.array(centres)


@pytest.mark.parametrize("levels", [6, 14, 30])
def test_deep_trees_are_exact_or_refused(hip_ctx, levels):
    """A tree whose worst-case traversal stack exceeds the 64 entries the
    traversal keeps is refused at build time (a silent overflow would drop
    subtrees); every tree that builds matches the brute force on rays aimed
    at the clumps of every scale."""
    b, centres = nested_clumps(levels)
    for builder in (F.RAD_BVH_DEVICE, F.RAD_BVH_HOST):
        try:
            g = hip.Scene.from_builder(hip_ctx, b, builder=builder)
        except hip.RadError as e:
            print(f"levels {levels} builder {builder}: refused ({e})", flush=True)
            assert e.status == 4 and "stack" in str(e)  # RAD_ERR_UNSUPPORTED
            continue
        info = g.info()
        print(f"levels {levels} builder {builder}: depth {info.bvh_depth}, stack need {info.bvh_stack_need}",
              flush=True)
        assert info.bvh_stack_need <= 64
        if levels <= 6:
            assert info.bvh_stack_need <= 3 * (info.bvh_depth - 1)
        o = O.OracleScene(b)
        rng = np.random.default_rng(levels)
        n = 6000
        rays = np.zeros(n, hip.RAY_DTYPE)
        org = rng.normal(size=(n, 3))
        org = 3.0 * org / np.linalg.norm(org, axis=1, keepdims=True)
        tgt = centres[rng.integers(len(centres), size=n)] + rng.normal(0, 1e-3, (n, 3))
        d = tgt - org
        rays["o"] = org.astype(np.float32)
        rays["d"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
        rays["tmax"] = 3e38
        check_parity(o, rays, g.closest(rays), o.closest(rays, brute=True))
        assert np.array_equal(g.occluded(rays).astype(bool), o.occluded(rays, brute=True).astype(bool))


def rays_along_z(extent, n, seed):
    """Rays from z = -1 through points of z = 0 with x and y of up to `extent`, with slopes of its size: exact to
    float precision however small it is (components below 1e-18 are left out: the traversal raises them to that)."""
    rng = np.random.default_rng(seed)
    rays = np.zeros(n, hip.RAY_DTYPE)
    to, d = rng.uniform(-extent, extent, (n, 2)), rng.uniform(0.01, 1, (n, 2)) * rng.choice([-extent, extent], (n, 2))
    rays["o"] = np.concatenate([to - d, np.full((n, 1), -1.0)], 1)
    rays["d"] = np.concatenate([d, np.ones((n, 1))], 1)
    rays["tmax"] = 3e38
    return rays


@pytest.mark.parametrize("leaf", [33, 255, 256, 603])
def test_leaf_at_the_host_builders_depth_limit(hip_ctx, leaf):
    """A leaf of 255 primitives is traversed; a larger one is refused before anything of the scene changes, so the
    tree it had stays in use."""
    tris = shrinking_sequence(leaf)
    b = mesh_scene(tris)
    o = O.OracleScene(b)
    rays = rays_along_z(1.2 * float(np.abs(tris[60:]).max()), 4000, leaf)
    hb = o.closest(rays, brute=True)
    assert 0.01 < (hb["geom"] != 0xFFFFFFFF).mean() < 0.99
    g = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_DEVICE)
    before = g.closest(rays)
    check_parity(o, rays, before, hb)
    if leaf <= 255:
        g.build_bvh(F.RAD_BVH_HOST)
        r = g.bvh_check()
        assert r.max_leaf == leaf and r.quantized_box_violations == 0 and r.leaf_box_violations == 0
        assert r.structure_errors == 0 and r.unreferenced_or_repeated == 0
    else:
        with pytest.raises(hip.RadError, match=f"leaf of {leaf} ") as e:
            g.build_bvh(F.RAD_BVH_HOST)
        assert e.value.status == 1  # RAD_ERR_INVALID_ARG
        assert np.array_equal(g.closest(rays), before)
    check_parity(o, rays, g.closest(rays), hb)
    assert np.array_equal(g.occluded(rays).astype(bool), hb["geom"] != 0xFFFFFFFF)


def test_failed_rebuild(hip_ctx):
    """A rebuild refused for its arguments leaves the tree in use; one that fails after it has written to the tree's
    buffers (here: a stack need above 64) leaves the scene without one until a build succeeds."""
    b, centres = nested_clumps(43)
    g = hip.Scene.from_builder(hip_ctx, b, builder=F.RAD_BVH_DEVICE)
    assert g.info().bvh_stack_need == 64  # the deepest that is traversed
    rng = np.random.default_rng(1)
    rays = np.zeros(6000, hip.RAY_DTYPE)
    org = rng.normal(size=(6000, 3))
    org = 3.0 * org / np.linalg.norm(org, axis=1, keepdims=True)
    d = centres[rng.integers(len(centres), size=6000)] + rng.normal(0, 1e-3, (6000, 3)) - org
    rays["o"], rays["d"], rays["tmax"] = org, d / np.linalg.norm(d, axis=1, keepdims=True), 3e38
    hb = O.OracleScene(b).closest(rays, brute=True)
    check_parity(O.OracleScene(b), rays, g.closest(rays), hb)
    for kw in ({"max_leaf": 17}, {"builder": 7}):
        with pytest.raises(hip.RadError) as e:
            g.build_bvh(**kw)
        assert e.value.status == 1
        check_parity(O.OracleScene(b), rays, g.closest(rays), hb)
    with pytest.raises(hip.RadError, match="stack") as e:
        g.build_bvh(F.RAD_BVH_HOST)
    assert e.value.status == 4
    for query in (g.closest, g.occluded, lambda r: g.render(b.render_desc(spp=1, seed=1)), lambda r: g.bvh_check()):
        with pytest.raises(hip.RadError) as e:
            query(rays)
        assert e.value.status == 7  # RAD_ERR_STATE
    g.build_bvh(F.RAD_BVH_DEVICE)
    check_parity(O.OracleScene(b), rays, g.closest(rays), hb)


@pytest.mark.parametrize("copies", [1, 6])
@pytest.mark.parametrize("n", [60, 1500, 1700, 9000, 14000])
def test_small_and_large_tree_paths(hip_ctx, n, copies):
    """Triangle counts on both sides of the sizes at which the traversal's nodes are made on the host (host builder),
    by one block and level by level: hits, ties between copies and the tree's structure."""
    rng = np.random.default_rng(n)
    t = rng.uniform(-1, 1, (n // copies, 1, 3)) + rng.normal(0, 0.1, (n // copies, 3, 3))
    b = mesh_scene(np.concatenate([t] * copies))
    o = O.OracleScene(b)
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, 2000, n)
    hb = o.closest(rays, brute=True)
    for builder in (F.RAD_BVH_DEVICE, F.RAD_BVH_HOST):
        for max_leaf in (1, 4, 16):
            g = hip.Scene.from_builder(hip_ctx, b, builder=builder, max_leaf=max_leaf)
            r = g.bvh_check()
            assert r.structure_errors == 0 and r.unreferenced_or_repeated == 0 and r.leaf_box_violations == 0
            assert r.child_box_violations == 0 and r.quantized_box_violations == 0
            h = g.closest(rays)
            check_parity(o, rays, h, hb)
            g.build_bvh(builder, max_leaf)  # again, into the buffers that are there
            assert np.array_equal(h, g.closest(rays))
