"""GPU: the deferred composite's arithmetic where its result is known.

A variance shadow map cleared to a huge or infinite distance ("no occluder")
lights, as the division by the smoothstep's window says (+inf, clamped to 1),
and so does a variance whose reciprocal FP32 cannot hold. The powers are seen
one at a time, through scenes whose other factors are exact: the gamma is
within 1.32 ulp of the 64-bit power of its FP32 argument, which is what the
library's powf reaches here over all significands, and (n.h)^20 within 0.51 ulp
(half for the rounding to FP32). What passes through the gamma has its relative
error divided by 2.2; an ulp is at most 2^-23 of its number."""
import numpy as np
import pytest

import mlgi

pytestmark = pytest.mark.gpu

F = np.float32
GAMMA = float(F(1) / F(2.2))
POWF = 1.32
ULP = 2.0 ** -23


def scene(w, h, **kw):
    """Every pixel at the origin, seen and lit along z; light (0, 0, 6)."""
    n = np.zeros((h, w, 3), F)
    n[..., :2], n[..., 2] = 0.5, 1.0
    i = dict(depth=np.full((h, w), 0.5, F), normal=n, diffuse=np.zeros((h, w, 3), F), gi=np.zeros((h, w, 3), F),
             specular=np.zeros((h, w, 3), F), vsm=np.full((2, 2, 2), 1e6, F))
    i["vsm"][..., 1] = 1e12
    i.update({k: v for k, v in kw.items() if k in i})
    m = np.zeros((4, 4), F)
    m[3, 3] = 1.0
    b = np.zeros((4, 4), F)  # column-major: the map's middle, between its four texels
    b[3, 0] = b[3, 1] = 0.5
    b[3, 3] = 1.0
    p = dict(vp_inv=m.ravel(), biased_light_vp=b.ravel(), eye=(0, 0, 4), light_pos=(0, 0, 6), inv_light_dir=(0, 0, 1),
             light_intensity=1.0, exposure=1.0)
    p.update({k: v for k, v in kw.items() if k in p})
    return i, p


def run(ctx, i, p):
    h, w = i["depth"].shape
    dev = {k: ctx.upload(np.ascontiguousarray(v)) for k, v in i.items()}
    out = ctx.empty((h, w, 3), np.float32)
    mlgi.deferred_composite(ctx, dev["depth"], dev["normal"], dev["diffuse"], dev["gi"], dev["vsm"], out,
                            specular=dev["specular"], **p)
    ctx.sync()
    return out.numpy()


def ulps(got, want):
    return np.abs(got.astype(np.float64) - want) / np.spacing(want.astype(F)).astype(np.float64)


@pytest.mark.parametrize("first,second", [(1e30, np.inf), (3.5e35, np.inf), (3e38, np.inf),
                                          (np.finfo(F).max, np.finfo(F).max), (np.inf, np.inf), (0.0, 1.5e38),
                                          (0.0, 3e38), (1e18, 2e38)])
def test_huge_moments_light(ctx, first, second):
    print(f"[composite] moments {first} {second}", flush=True)
    grey = np.full((5, 66, 3), 0.5, F)
    i, p = scene(66, 5, diffuse=grey, specular=grey)
    want = run(ctx, i, p)
    i["vsm"][..., 0], i["vsm"][..., 1] = first, second
    assert want.min() > 0.2
    assert np.array_equal(run(ctx, i, p), want)


def test_gamma(ctx):
    print("[composite] gamma", flush=True)
    rng = np.random.default_rng(3)
    g = np.exp(rng.uniform(np.log(1e-36), np.log(1e6), (64, 512, 3))).astype(F)
    out = run(ctx, *scene(512, 64, diffuse=np.ones_like(g), gi=g, light_intensity=0.0))
    q = (g / (F(1) + g)).astype(np.float64)
    assert ulps(out, q ** GAMMA).max() <= POWF


def test_highlight(ctx):
    print("[composite] highlight", flush=True)
    e = np.random.default_rng(5).uniform(0.75, 1.0, (64, 512)).astype(F)
    nz = (e * F(2) - F(1)).astype(np.float64)
    n = np.full((64, 512, 3), 0.5, F)
    n[..., 2] = e
    scale = 2.0 ** -40
    out = run(ctx, *scene(512, 64, normal=n, specular=np.ones((64, 512, 3), F), exposure=scale))
    want = ((0.75 * nz ** 20 * scale) ** GAMMA)[..., None]
    # the power, its product with 0.75 (half an ulp) and the gamma
    assert (np.abs(out - want) / want).max() <= ((0.51 + 0.5) * GAMMA + POWF) * ULP
