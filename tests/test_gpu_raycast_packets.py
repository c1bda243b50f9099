"""GPU: the packet ray casters against the host renderer, bit for bit, where a
packet can go wrong: images that do not fill its tiles, both sides of the
line between the two packet forms (2^18 texels), scenes of a single leaf and
of many nodes, rays along an axis (zero direction components), and cameras
outside the scene's box (rays that enter it late, miss it, or end before
it)."""
import numpy as np
import pytest

import mlgi
from mlgi import workloads as W

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (3, 5), (9, 7), (66, 33), (511, 512), (512, 512), (641, 410)]


def camera(kind, aspect):
    cam = mlgi.Camera.default(aspect)
    if kind == "axis":
        cam.eye, cam.center = (5.0, 5.0, 5.0), (5.0, 5.0, 0.0)
    elif kind == "outside":
        cam.eye, cam.center = (-3.0, 14.0, 21.0), (5.0, 5.0, 5.0)
    elif kind == "far":
        cam.eye, cam.center = (40.0, 30.0, 5.0), (5.0, 5.0, 5.0)
    return cam


@pytest.mark.parametrize("kind", ["inside", "axis", "outside", "far"])
@pytest.mark.parametrize("n_random", [0, 3, 4_000])
def test_packets_equal_host(ctx, n_random, kind):
    scene = W._scene(2, n_random)
    dev = scene.upload(ctx)
    for w, h in SIZES:
        print(f"[packets] {n_random} {kind} {w}x{h}", flush=True)
        cam = camera(kind, w / h)
        want = scene.render_gbuffer(cam, w, h) + scene.render_rsm(cam, w, h)[:3] + scene.render_surface(cam, w, h)
        d, n = ctx.empty((h, w), np.float32), ctx.empty((h, w, 3), np.float32)
        dev.render_gbuffer(cam, d, n)
        got = [d.numpy(), n.numpy()]
        a, b, c = ctx.empty((h, w, 3), np.float32), ctx.empty((h, w, 3), np.float32), ctx.empty((h, w), np.float32)
        dev.render_rsm(cam, a, b, c)
        got += [a.numpy(), b.numpy(), c.numpy()]
        alb, mom = ctx.empty((h, w, 3), np.float32), ctx.empty((h, w, 2), np.float32)
        dev.render_surface(cam, alb, mom)
        got += [alb.numpy(), mom.numpy()]
        for g, x in zip(got, want):
            assert np.array_equal(g, x)
        for arr in (d, n, a, b, c, alb, mom):
            arr.free()
    dev.close()
