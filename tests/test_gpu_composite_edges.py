"""GPU: the deferred composite at the edges of its 64 x 4 tiles and of its
arithmetic: albedos and irradiances of 0, denormals, tiny and huge values (whose
powers leave FP32's range), infinities, NaN and negative ones, cameras whose w
is 0, and lights beyond the distance where the VSM's 0.001 window rounds away.
The scene is fully lit (VSM moments beyond every distance), so that no shadow
edge amplifies rounding. The reference is the same formula in numpy FP32, whose
powers are within an ulp: where the colour is a normal float, outputs agree
within 3e-6 relative (two powers of at most 2 ulp, some ten roundings of 2^-24,
and the highlight's (n.h)^20, whose FP32 argument is good to 2^-22, together
below (40 x 2^-24 + 20 x 2^-22) / 2.2 = 3.2e-6 for a colour that is all
highlight, under half of that here), below that within 1e-15, and an output of
exactly 0 (an infinite or NaN colour, no light) is exactly 0."""
import numpy as np
import pytest

import mlgi

pytestmark = pytest.mark.gpu


def inputs(w, h, seed, light_far):
    rng = np.random.default_rng(seed)
    f = np.float32
    n = rng.normal(size=(h, w, 3))
    n[..., 2] = np.abs(n[..., 2]) + 0.5
    n /= np.linalg.norm(n, axis=-1, keepdims=True)
    i = dict(depth=rng.uniform(0.2, 0.8, (h, w)).astype(f), normal=(n * 0.5 + 0.5).astype(f),
             diffuse=rng.uniform(0, 1, (h, w, 3)).astype(f), specular=rng.uniform(0, 0.2, (h, w, 3)).astype(f),
             gi=rng.uniform(0, 2, (h, w, 3)).astype(f), occlusion=rng.uniform(0.3, 1, (h, w)).astype(f),
             vsm=np.full((8, 8, 2), 0, f))
    odd = [0.0, 1e-45, 1e-39, 1e-30, 1e-10, 0.75, np.nextafter(f(0.75), f(0)), 1.0, 1.5, 1e3, 1e12, 1e25, -1.0, np.inf,
           np.nan]
    flat = i["diffuse"].reshape(-1)
    flat[:len(odd)] = odd
    i["gi"].reshape(-1)[20:20 + len(odd)] = odd
    z = 3e5 if light_far else 6.0
    i["vsm"][..., 0] = 40 * z  # also where a corner's taps blend a quarter of it with the border's 0
    i["vsm"][..., 1] = 1600.0 * z * z
    blvp = np.zeros((4, 4), f)
    blvp[0, 0] = blvp[1, 1] = 0.5
    blvp[0, 3] = blvp[1, 3] = 0.5
    blvp[2, 2] = blvp[3, 3] = 1.0
    ld = np.array([-0.3, 0.2, -1.0])
    p = dict(vp_inv=np.eye(4, dtype=f).T.ravel(), biased_light_vp=blvp.T.ravel(), eye=(0.1, 0.2, 4.0),
             light_pos=(0.3, -0.2, z), inv_light_dir=-ld / np.linalg.norm(ld), light_intensity=1.7, exposure=1.3)
    return i, p


def run(ctx, i, p):
    h, w = i["depth"].shape
    dev = {k: ctx.upload(v) for k, v in i.items()}
    out = ctx.empty((h, w, 3), np.float32)
    mlgi.deferred_composite(ctx, dev["depth"], dev["normal"], dev["diffuse"], dev["gi"], dev["vsm"], out,
                            specular=dev["specular"], occlusion=dev["occlusion"], **p)
    ctx.sync()
    return out.numpy()


def ref(i, p):
    f = np.float32
    with np.errstate(all="ignore"):
        h, w = i["depth"].shape
        x = np.broadcast_to(((np.arange(w, dtype=f) + f(0.5)) / f(w) * f(2) - f(1))[None, :], (h, w))
        y = np.broadcast_to(((np.arange(h, dtype=f) + f(0.5)) / f(h) * f(2) - f(1))[:, None], (h, w))
        ndc = [x, y, i["depth"] * f(2) - f(1), np.ones((h, w), f)]
        m = np.asarray(p["vp_inv"], f).reshape(4, 4)  # [column][row]
        r = [sum((m[c, k] * ndc[c] for c in range(1, 4)), m[0, k] * ndc[0]) for k in range(4)]
        pos = [r[k] / r[3] for k in range(3)]
        n = [i["normal"][..., k] * f(2) - f(1) for k in range(3)]
        light = [f(v) for v in p["inv_light_dir"]]

        def unit(v):
            l = np.sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2])
            return [c / l for c in v]
        view = unit([f(e) - c for e, c in zip(p["eye"], pos)])
        half = unit([a + b for a, b in zip(light, view)])
        ndl = n[0] * light[0] + n[1] * light[1] + n[2] * light[2]
        ndh = n[0] * half[0] + n[1] * half[1] + n[2] * half[2]
        power = lambda v, e: np.where(v > 0, np.power(np.where(v > 0, v, f(1)), f(e)), f(0)).astype(f)  # noqa: E731
        spec = power(np.maximum(ndh, f(0)), 20.0)
        dif, spc = power(i["diffuse"], 2.2), power(i["specular"], 2.2)
        occ = i["occlusion"][..., None]
        col = (i["gi"] * dif * occ + dif * np.maximum(ndl, f(0))[..., None] * f(p["light_intensity"])
               + f(0.75) * spc * spec[..., None]) * f(p["exposure"])
        return power(col / (f(1) + col), f(1) / f(2.2))


@pytest.mark.parametrize("light_far", [False, True])
@pytest.mark.parametrize("w,h", [(63, 3), (64, 4), (65, 5), (128, 9), (17, 2)])
def test_composite_edges(ctx, w, h, light_far):
    print(f"[composite] edges {w}x{h} far={light_far}", flush=True)
    i, p = inputs(w, h, w + h, light_far)
    got, want = run(ctx, i, p).astype(np.float64), ref(i, p).astype(np.float64)
    assert np.isfinite(got).all()
    plain = want > float(np.finfo(np.float32).tiny) ** (1 / 2.2)
    assert (np.abs(got - want)[plain] / want[plain]).max() <= 3e-6
    assert (np.abs(got - want)[~plain] <= 1e-15).all()
    assert (got[want == 0] == 0).all()


def test_zero_w_has_no_infinity(ctx):
    i, p = inputs(64, 4, 1, False)
    m = np.eye(4, dtype=np.float32)
    m[3, 3] = 0.0  # inverse(P*V) with w = 0 everywhere
    p["vp_inv"] = m.T.ravel()
    assert np.isfinite(run(ctx, i, p)).all()
