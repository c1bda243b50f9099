"""The ray caster's tree against its traversal stack (CPU only). The device's
packets keep their pending children in 128 entries without a check, so the
build must bound them: the tree of area splits is taken where it fits, else one
of median splits and whole levels, at most 7 per three levels; neither fitting
is an error. Both trees render the same texels."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

import mlgi

SRC = Path(__file__).with_name("bvh_stack.cpp")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("bvh") / "libbvh.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", str(SRC), "-o", str(so),
                    "-lpthread"], check=True)
    return C.CDLL(str(so))


def render(lib, scene, w, h):
    cam = mlgi.Camera.default(w / h).to_c()
    depth, normal = np.empty((h, w), np.float32), np.empty((h, w, 3), np.float32)
    assert lib.mlgi_scene_render_gbuffer(scene, C.byref(cam), w, h, 2, depth.ctypes.data_as(C.c_void_p),
                                         normal.ctypes.data_as(C.c_void_p)) == 0
    return depth, normal


@pytest.mark.parametrize("n_random", [5, 4_000, 40_000])
def test_tree_by_levels(lib, n_random):
    scene = C.c_void_p()
    assert lib.mlgi_scene_create(C.c_uint64(2), n_random, C.byref(scene)) == 0
    area = lib.max_pending(scene)
    want = render(lib, scene, 97, 61)
    assert lib.rebuild(scene, area + 1) == 1 and lib.max_pending(scene) == area  # it just fits
    n = n_random + 12
    binary = int(np.ceil(np.log2(n / 4))) + 2
    levels = 7 * -(-binary // 3)
    assert lib.rebuild(scene, area) == 1  # too small for that tree
    assert lib.max_pending(scene) < area and lib.max_pending(scene) <= levels
    assert all(np.array_equal(g, w) for g, w in zip(render(lib, scene, 97, 61), want))
    assert lib.rebuild(scene, 2) == 0
    lib.mlgi_scene_destroy(scene)


def test_levels_fit_the_stack_for_any_count():
    assert 7 * -(-31 // 3) < 128
