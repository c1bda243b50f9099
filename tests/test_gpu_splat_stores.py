"""GPU: tiles stored write-through (launches of small atlases) and as a stream
(176 MiB and more of tiles in a launch): the same atlas as the point-major
splat's atomics give, alone and in batches on both sides of the line, and the
same ISM."""
import numpy as np
import pytest

import mlgi
from mlgi import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_vpl,atlas,frames", [(4096, 4096, 2), (4096, 4096, 3), (1024, 1024, 44), (16384, 8192, 1)])
def test_tile_stores(ctx, n_vpl, atlas, frames):
    print(f"[splat] stores N={n_vpl} atlas={atlas} frames={frames}", flush=True)
    wl = W.WORKLOADS["tiny"].with_(n_vpl=n_vpl, interleave=4, atlas_side=atlas, n_points=20_000, levels=3)
    inp = W.build_inputs(wl)
    rsm = mlgi.rsm_desc(ctx.upload(inp.rsm_diffuse), ctx.upload(inp.rsm_normal), ctx.upload(inp.rsm_depth), inp.inv_bvp)
    pts = mlgi.points_desc(ctx.upload(inp.points), ctx.upload(inp.bin_offsets))
    gb = mlgi.gbuffer_desc(ctx.upload(inp.gb_depth), ctx.upload(inp.gb_normal), inp.vp_inv)
    images = []
    for block in (256, 0):
        p = wl.params()
        p.splat_block = block
        one = mlgi.GIStage(ctx, p, n_vpl, wl.width, wl.height)
        one.process(rsm, pts, gb)
        ctx.sync()
        images.append((one.ism.softrender.numpy(), one.ism.pushpull_result.numpy()))
    (want, ism), (got, got_ism) = images
    assert (want != 0xFFFFFFFF).any()
    assert np.array_equal(got, want) and np.array_equal(got_ism, ism)
    stages = [mlgi.GIStage(ctx, p, n_vpl, wl.width, wl.height) for _ in range(frames)]
    b = mlgi.Batch(ctx, [(st, rsm, pts, gb) for st in stages])
    b.run()
    ctx.sync()
    for st in stages:
        assert np.array_equal(st.ism.softrender.numpy(), want) and np.array_equal(st.ism.pushpull_result.numpy(), ism)
    b.close()
