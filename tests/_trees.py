"""Triangle sets that lead the tree builders to their limits."""
import numpy as np

from radiantiumplusplus_amd import scenes


def bounds_of(tris):
    """(n, 6) float32 boxes of (n, 3, 3) triangles."""
    t = np.asarray(tris, np.float32)
    return np.ascontiguousarray(np.concatenate([t.min(1), t.max(1)], 1))


def shrinking_sequence(cluster, top=1e17, ratio=34.0, seed=0):
    """Twenty triangles on each axis at top, top / ratio, ... and `cluster` triangles near the origin: the host
    builder's splits take one triangle each off the rest, so its 60 levels end in a leaf that is the cluster."""
    rng = np.random.default_rng(seed)
    out = []
    for a in range(3):
        for i in range(20):
            s = top / ratio**i
            c = np.zeros(3)
            c[a] = s
            out.append([c, c + [1e-3 * s, 0, 0], c + [0, 1e-3 * s, 1e-3 * s]])
    s = top / ratio**21
    near = rng.uniform(-1, 1, (cluster, 1, 3)) * s + rng.normal(0, 0.01 * s, (cluster, 3, 3))
    return np.concatenate([np.array(out), near]).astype(np.float32)


def mesh_scene(tris):
    b = scenes.SceneBuilder()
    p = np.asarray(tris, np.float32).reshape(-1, 3)
    b.mesh(p, np.arange(len(p), dtype=np.uint32), bsdf=b.diffuse(0.5))
    b.skybox(1.0)
    b.set_camera(8, 8, 45, origin=(0, 0, -5), target=(0, 0, 0), far=100)
    return b
