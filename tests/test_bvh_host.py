"""The host tree builder's leaves, without a device."""
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
    return C.CDLL(so)


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
