"""GPU: cameras whose rays are infinite, NaN or barely resolved in FP64 (no far
plane, a plane beyond the doubles' reach, a camera at its own centre). Both
packet forms (33 x 17 texels and 513 x 512) give the host renderer's texels;
rays that are not finite hit nothing. test_box_rays.py shows on the CPU that
none of these rays enters an unused child."""
from dataclasses import replace

import numpy as np
import pytest

import mlgi
from mlgi import workloads as W

pytestmark = pytest.mark.gpu

CAMERAS = {
    "no far plane": dict(z_far=float("inf")),
    "far plane past FP64": dict(z_far=1e20),
    "far plane 1e14": dict(z_far=1e14),
    "along the diagonal": dict(eye=(2, 2, 2), center=(3, 3, 3), z_far=1e14),
    "looks at its eye": dict(center=(5, 5, 9)),
    "nan": dict(eye=(float("nan"), 5, 9)),
}


@pytest.mark.parametrize("kind", CAMERAS)
@pytest.mark.parametrize("w,h", [(33, 17), (513, 512)])
def test_degenerate_cameras_equal_host(ctx, w, h, kind):
    print(f"[packets] {kind} {w}x{h}", flush=True)
    scene = W._scene(2, 500)
    dev = scene.upload(ctx)
    cam = replace(mlgi.Camera.default(w / h), **CAMERAS[kind])
    d, n = ctx.empty((h, w), np.float32), ctx.empty((h, w, 3), np.float32)
    dev.render_gbuffer(cam, d, n)
    for got, want in zip((d, n), scene.render_gbuffer(cam, w, h)):
        assert np.array_equal(got.numpy(), want, equal_nan=True)
    dev.close()
