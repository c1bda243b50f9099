"""The packet ray casters' FP32 box tests (CPU only). A packet follows every
child reference whose box some ray enters, so no ray at all may enter the box
of an unused child, whose reference names no node: not one of a camera without
a far plane, nor of one that looks at its own eye, whose rays are infinite or
NaN (and enter no box at all, as in the host renderer)."""
import ctypes as C
import subprocess
from dataclasses import replace
from pathlib import Path

import pytest

import mlgi
from mlgi import _native as N

SRC = Path(__file__).with_name("box_rays.cpp")
INF, BIG = float("inf"), 3e38


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("box") / "libbox.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", str(SRC), "-o", str(so),
                    "-lpthread"], check=True)
    L = C.CDLL(str(so))
    L.unused_hits.argtypes = [C.c_void_p, C.POINTER(N.Camera), C.c_int, C.c_int, C.POINTER(C.c_long)]
    L.unused_hits.restype = C.c_long
    return L


CAMERAS = {
    "default": {},
    "no far plane": dict(z_far=INF),
    "far plane past FP64": dict(z_far=1e20),
    "along the diagonal": dict(eye=(2, 2, 2), center=(3, 3, 3), z_far=1e30, z_near=1e14),
    "largest planes": dict(eye=(2, 2, 2), center=(3, 3, 3), z_near=1e22, z_far=BIG),
    "looks at its eye": dict(center=(5, 5, 9)),
    "nan": dict(eye=(float("nan"), 5, 9)),
    "infinitely far": dict(eye=(INF, 5, 9)),
    "far away": dict(eye=(-BIG, 5, 9)),
    "no opening": dict(fovy_deg=0.0),
    "flat": dict(z_near=1.0, z_far=1.0),
}


@pytest.mark.parametrize("kind", CAMERAS)
@pytest.mark.parametrize("n_random", [0, 3, 500])
def test_unused_children_are_never_entered(lib, n_random, kind):
    scene, stray = C.c_void_p(), C.c_long(0)
    assert lib.mlgi_scene_create(C.c_uint64(2), n_random, C.byref(scene)) == 0
    cam = replace(mlgi.Camera.default(1.0), **CAMERAS[kind]).to_c()
    unused = lib.unused_hits(scene, C.byref(cam), 17, 17, C.byref(stray))
    lib.mlgi_scene_destroy(scene)
    assert (unused, stray.value) == (0, 0)
