"""GPU: the blur at the edges of its 64 x 16 tiles and two-pixel runs, bit for
bit against the oracle's FP32 instantiation: images of one pixel, one row, one
column, one short of a tile, a tile, one past it; flat geometry (every weight
at work), unrelated normals and depth steps (weights of 0), black and bright
pixels."""
import numpy as np
import pytest

import mlgi
import oracle

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 40), (70, 1), (2, 3), (63, 15), (64, 16), (65, 17), (66, 31), (129, 33), (200, 50)]


@pytest.mark.parametrize("flat", [True, False])
def test_blur_edges(ctx, flat):
    proj = np.ascontiguousarray(mlgi.Camera.default(1.5).matrices()[1], np.float32)
    for w, h in SIZES:
        print(f"[blur] edges {w}x{h} flat={flat}", flush=True)
        rng = np.random.default_rng(w * 1000 + h)
        f = np.float32
        gi = rng.uniform(0, 2, (h, w, 3)).astype(f)
        gi[rng.random((h, w)) < 0.1] = 0
        gi[rng.random((h, w)) < 0.05] *= f(1e4)
        n = np.tile(np.array([0.0, 0.6, 0.8]), (h, w, 1)) + (0.02 if flat else 0.5) * rng.normal(size=(h, w, 3))
        n /= np.linalg.norm(n, axis=-1, keepdims=True)
        normal = (n * 0.5 + 0.5).astype(f)
        depth = (0.99 + (1e-4 if flat else 5e-3) * rng.uniform(-1, 1, (h, w))).astype(f)
        st = mlgi.GIStage(ctx, mlgi.default_params(atlas_side=64), 16, w, h)
        st.gi_buffer.copy_from(gi)
        gb = mlgi.gbuffer_desc(ctx.upload(depth), ctx.upload(normal), np.eye(4, dtype=f).ravel())
        st.blur(gb, proj)
        ctx.sync()
        assert np.array_equal(st.gi_blur_final.numpy(), oracle.gi_blur(gi, normal, depth, proj, np.float32)), (w, h)
