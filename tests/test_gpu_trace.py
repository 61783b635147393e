"""Edges of the 8-wide traversal: batches of every share of a wave's lanes,
leaves from one primitive to more than a node's own 32, 64-bit node addresses,
hits behind the origin and exact ties."""
import numpy as np
import pytest

import _oracle as O
from radiantiumplusplus_amd import _ffi as F
from radiantiumplusplus_amd import hip, scenes
from test_gpu_intersect import check_parity, ray_batch

pytestmark = pytest.mark.gpu


def soup(n, size, seed, spread=1.0):
    """n random triangles of about `size` in a cube of side 2 * spread."""
    rng = np.random.default_rng(seed)
    p = rng.uniform(-spread, spread, (n, 1, 3)) + rng.normal(0, size, (n, 3, 3))
    b = scenes.SceneBuilder()
    b.mesh(p.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32), bsdf=b.diffuse(0.5))
    b.skybox(1.0)
    b.set_camera(8, 8, 45, origin=(0, 0, -5), target=(0, 0, 0), far=100)
    return b


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4095, 16 * 4096, 16 * 4096 + 1, 150001])
def test_batch_sizes(hip_ctx, n):
    """Batches around a wave's smallest share, a full wave and shares of more rays than lanes."""
    b = soup(500, 0.1, 1)
    o = O.OracleScene(b)
    g = hip.Scene.from_builder(hip_ctx, b)
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, n, n)
    hb = o.closest(rays, brute=True)
    check_parity(o, rays, g.closest(rays), hb)
    assert np.array_equal(g.occluded(rays).astype(bool), hb["geom"] != 0xFFFFFFFF)


@pytest.mark.parametrize("builder", [F.RAD_BVH_DEVICE, F.RAD_BVH_HOST])
@pytest.mark.parametrize("max_leaf", [1, 2, 7, 8, 9, 15, 16])
def test_leaf_sizes(hip_ctx, builder, max_leaf):
    """Triangles that overlap so much that leaves fill: siblings with up to 64
    primitives, of which a node holds 32 and the rest get nodes of their own."""
    b = soup(700, 0.8, 2)
    o = O.OracleScene(b)
    g = hip.Scene.from_builder(hip_ctx, b, builder=builder, max_leaf=max_leaf)
    r = g.bvh_check()
    assert r.structure_errors == 0 and r.unreferenced_or_repeated == 0 and r.leaf_box_violations == 0
    assert r.child_box_violations == 0 and r.quantized_box_violations == 0
    assert r.max_leaf <= max_leaf
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, 3000, max_leaf)
    hb = o.closest(rays, brute=True)
    check_parity(o, rays, g.closest(rays), hb)
    assert np.array_equal(g.occluded(rays).astype(bool), hb["geom"] != 0xFFFFFFFF)


def test_far_node_addresses(hip_ctx, monkeypatch):
    """The kernels for trees of 4 GiB or more give the same hits and images."""
    b = scenes.many_balls(seed=4, n_spheres=40, width=48, height=32)
    near = hip.Scene.from_builder(hip_ctx, b)
    monkeypatch.setenv("RAD_TRACE_FAR", "1")
    far = hip.Scene.from_builder(hip_ctx, b)
    rays = ray_batch(np.array([-6.0, 0, -6]), np.array([6.0, 6, 6]), 5000, 3)
    assert np.array_equal(near.closest(rays), far.closest(rays))
    assert np.array_equal(near.occluded(rays), far.occluded(rays))
    d = b.render_desc(spp=4, seed=2)
    assert np.array_equal(near.render(d)[0], far.render(d)[0])


def test_hits_behind_the_origin(hip_ctx):
    """A negative tmin admits hits behind the origin; the closest is the smallest t."""
    b = soup(60, 0.5, 5)
    o = O.OracleScene(b)
    g = hip.Scene.from_builder(hip_ctx, b)
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, 4000, 9)
    rays["tmin"] = -3.0
    hb = o.closest(rays, brute=True)
    assert (hb["t"][hb["geom"] != 0xFFFFFFFF] < 0).any()
    check_parity(o, rays, g.closest(rays), hb)


def test_ties_do_not_depend_on_the_batch(hip_ctx):
    """Coincident triangles: which of them a ray reports is a property of the
    scene, not of the rays traced with it."""
    rng = np.random.default_rng(6)
    p = rng.uniform(-1, 1, (200, 1, 3)) + rng.normal(0, 0.3, (200, 3, 3))
    p = np.concatenate([p, p, p]).reshape(-1, 3).astype(np.float32)
    b = scenes.SceneBuilder()
    b.mesh(p, np.arange(len(p), dtype=np.uint32), bsdf=b.diffuse(0.5))
    b.skybox(1.0)
    b.set_camera(8, 8, 45, origin=(0, 0, -5), target=(0, 0, 0), far=100)
    g = hip.Scene.from_builder(hip_ctx, b)
    rays = ray_batch(np.array([-2.0, -2, -2]), np.array([2.0, 2, 2]), 6000, 8)
    whole = g.closest(rays)
    order = rng.permutation(len(rays))
    assert np.array_equal(whole[order], g.closest(rays[order]))
    assert np.array_equal(whole[100:163], g.closest(rays[100:163]))
    assert np.array_equal(whole[7:8], g.closest(rays[7:8]))


@pytest.mark.parametrize("builder", [F.RAD_BVH_DEVICE, F.RAD_BVH_HOST])
@pytest.mark.parametrize("axis", [False, True])
def test_ties_between_nodes_do_not_depend_on_the_batch(hip_ctx, builder, axis):
    """A dozen copies of every triangle, one to a leaf, so that they lie in different nodes and are tested at
    different times; axis: in planes of constant z, where the boxes are flat.  Which copy a ray reports does not depend
    on what else is traced."""
    rng = np.random.default_rng(16)
    p = rng.uniform(-1, 1, (150, 1, 3)) + rng.normal(0, 0.3, (150, 3, 3))
    if axis:
        p[:, :, 2] = np.round(4 * p[:, :1, 2]) / 4
    p = np.concatenate([p] * 12).reshape(-1, 3).astype(np.float32)
    b = scenes.SceneBuilder()
    b.mesh(p, np.arange(len(p), dtype=np.uint32), bsdf=b.diffuse(0.5))
    b.skybox(1.0)
    b.set_camera(8, 8, 45, origin=(0, 0, -5), target=(0, 0, 0), far=100)
    g = hip.Scene.from_builder(hip_ctx, b, builder=builder, max_leaf=1)
    n = 200000
    rays = ray_batch(np.array([-2.0, -2, -2]), np.array([2.0, 2, 2]), n, 8)
    whole = g.closest(rays)
    assert (whole["geom"] != 0xFFFFFFFF).sum() > 10000
    for seed in range(3):
        order = np.random.default_rng(seed).permutation(n)
        got = g.closest(rays[order])
        assert np.array_equal(whole["t"][order], got["t"])
        assert (whole[order] != got).sum() == 0
    few = np.random.default_rng(9).permutation(n)[:3000]
    assert np.array_equal(whole[few], g.closest(rays[few]))


def test_hits_at_the_end_of_the_segment(hip_ctx):
    """A triangle accepts T <= |den| * tmax, whose right side may round up: a hit at t = T / |den| one ulp above tmax is
    a hit of both queries.  The rays are those that the brute force keeps with tmax one ulp below their t."""
    b = soup(300, 0.3, 11)
    o = O.OracleScene(b)
    g = hip.Scene.from_builder(hip_ctx, b)
    lo, hi = o.bounds()
    rays = ray_batch(lo, hi, 60000, 12)
    rays["tmax"] = 3e38
    h = o.closest(rays, brute=True)
    hit = h["geom"] != 0xFFFFFFFF
    rays, h = rays[hit], h[hit]
    rays["tmax"] = np.nextafter(h["t"], np.float32(0))
    kept = o.closest(rays, brute=True)
    end = (kept["geom"] != 0xFFFFFFFF) & (kept["t"] > rays["tmax"])
    assert end.sum() > 100
    check_parity(o, rays, g.closest(rays), kept)
    assert np.array_equal(g.occluded(rays).astype(bool), kept["geom"] != 0xFFFFFFFF)


@pytest.mark.parametrize("w,h", [(1, 1), (7, 5), (8, 8), (9, 17), (23, 3), (65, 31)])
def test_every_pixel_gets_its_samples(hip_ctx, w, h):
    """Images whose last tiles are partial: under a constant sky every pixel is
    the float32 running sum of its spp equal samples times 1/spp."""
    b = scenes.SceneBuilder()
    b.sphere(center=(0, 0, -50), radius=1.0, bsdf=b.diffuse(0.5))
    b.skybox((0.3, 0.7, 1.1))
    b.set_camera(w, h, 40, origin=(0, 0, 0), target=(0, 0, 1), far=100)
    b.set_render("path", spp=5, max_depth=4)
    img, _, st = hip.Scene.from_builder(hip_ctx, b).render(b.render_desc(spp=5, seed=1))
    acc = np.zeros(3, np.float32)
    for _ in range(5):
        acc = (acc + np.array([0.3, 0.7, 1.1], np.float32)).astype(np.float32)
    assert st.samples == 5 * w * h
    assert np.array_equal(img, np.broadcast_to((acc * np.float32(1 / np.float32(5))).astype(np.float32), img.shape))
