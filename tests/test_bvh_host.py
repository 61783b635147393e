"""The host tree builder and the 8-wide nodes made of its trees, without a device."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from radiantiumplusplus_amd import build
from _trees import bounds_of, shrinking_sequence

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("bvh") / "probe.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{os.path.join(build.ROOT, 'include')}", f"-I{build.CSRC}", os.path.join(HERE, "bvh_host_probe.cpp"),
                    "-o", so, "-lpthread"], check=True, capture_output=True)
    lib = C.CDLL(so)
    lib.probe_wide_broken.restype = C.c_int32
    return lib


def host_leaf(probe, tris, max_leaf=0):
    b, need = bounds_of(tris), C.c_uint32()
    return probe.probe_host_leaf(b.ctypes.data_as(C.c_void_p), len(b), max_leaf, C.byref(need)), need.value


@pytest.mark.parametrize("cluster", [255, 256, 603])
def test_leaf_at_the_depth_limit(probe, cluster):
    """After 60 levels the rest is one leaf, whatever max_leaf asks for, while the stack need stays at nothing.
    Leaves above kMaxLeafPrims must not reach the traversal's nodes: rad_hip_bvh_build refuses them."""
    assert host_leaf(probe, shrinking_sequence(cluster)) == (cluster, 0)
    assert probe.probe_max_leaf_prims() == 255


@pytest.mark.parametrize("max_leaf", [0, 1, 4, 15, 1000])
def test_leaves_of_ordinary_trees(probe, max_leaf):
    tris = np.random.default_rng(1).uniform(-1, 1, (3000, 1, 3)) + np.random.default_rng(2).normal(0, 0.3, (3000, 3, 3))
    assert host_leaf(probe, tris, max_leaf)[0] <= min(max_leaf or 4, 15)


def check_wide(errors, out):
    """No errors but a stack need above 64, which is at most the 4-wide tree's: what rad_hip_bvh_build bounds."""
    _, need, need4 = list(out)
    assert errors == (1 if need > 64 else 0) and need <= need4
    return need, need4


@pytest.mark.parametrize("inner,leaves", [(1, (16, 16, 16)), (1, (11, 11, 11)), (1, (10, 11, 11)), (1, (16, 16)), (2, (16, 16)),
                                          (2, (20, 20)), (1, (33,)), (2, (33, 1)), (1, (1, 255, 32)), (1, (255, 255, 255)),
                                          (1, (64, 32, 1)), (3, (97,)), (4, ()), (1, (32, 1))])
@pytest.mark.parametrize("length", [1, 2, 90])
def test_wide_nodes_of_a_chain(probe, inner, leaves, length):
    """Long paths of nodes whose leaves do not fit one 8-wide node: the leaves of the first form leave one inner child
    a level, a stack need of nothing, and must not ask the traversal for an entry a level (90 against its 64)."""
    out = (C.c_uint32 * 3)()
    errors = probe.probe_wide_chain(length, inner, (C.c_uint32 * 4)(*leaves), len(leaves), out)
    need, need4 = check_wide(errors, out)
    if inner == 1:
        assert need == need4 == 0


@pytest.mark.parametrize("max_leaf", [1, 2, 4, 8, 9, 15])
@pytest.mark.parametrize("n", [1, 2, 5, 33, 700, 20000])
def test_wide_nodes_of_host_trees(probe, n, max_leaf):
    rng = np.random.default_rng(n)
    b = bounds_of(rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0, 0.8 if n < 1000 else 0.05, (n, 3, 3)))
    out = (C.c_uint32 * 3)()
    check_wide(probe.probe_wide_host(b.ctypes.data_as(C.c_void_p), n, max_leaf, out), out)


@pytest.mark.parametrize("cluster", [33, 64, 65, 255, 603])
def test_wide_nodes_of_a_large_leaf(probe, cluster):
    b, out = bounds_of(shrinking_sequence(cluster)), (C.c_uint32 * 3)()
    check_wide(probe.probe_wide_host(b.ctypes.data_as(C.c_void_p), len(b), 0, out), out)


@pytest.mark.parametrize("what", range(8))
def test_structure_check_finds_errors(probe, what):
    """The check of rad_hip_bvh_check on trees with one mistake each: a plane of a child moved to the other side of its
    box (rectangle-like flat boxes among the primitives), wrong primitives, wrong children."""
    rng = np.random.default_rng(5)
    tris = rng.uniform(-1, 1, (300, 1, 3)) + rng.normal(0, 0.1, (300, 3, 3))
    tris[::3, :, 1] = tris[::3, :1, 1]
    b, found = bounds_of(tris), 0
    for x in range(0, 60, 7):
        for s in range(8):
            errors = probe.probe_wide_broken(b.ctypes.data_as(C.c_void_p), len(b), x, s, what)
            assert errors == -1 or errors > 0
            found += errors > 0
    assert found > 20
