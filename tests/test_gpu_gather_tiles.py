"""GPU: the final gather over ISM grids where the texel address can wrap (one
tile, all tiles on the atlas's border, few inner ones) and over tile shapes
and ragged images: every tile shape gives the same bits (the shape only changes
which pixels share a wave, and the culling is exact), single-frame and batched,
and the irradiance is within the forms' bars of the FP64 oracle."""
import numpy as np
import pytest

import mlgi
import oracle
from mlgi import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,bar", [(mlgi.PRECISION_FP32, 1e-4), (mlgi.PRECISION_MIXED, 2e-3)])
@pytest.mark.parametrize("n_vpl,interleave,atlas,size", [(1, 1, 64, (33, 17)), (4, 2, 64, (40, 30)), (16, 4, 256, (97, 61)),
                                                         (64, 2, 256, (70, 45)), (192, 4, 512, (131, 75))])
def test_tile_shapes_and_wraps(ctx, n_vpl, interleave, atlas, size, precision, bar):
    print(f"[gather] N={n_vpl} I={interleave} atlas={atlas} {size} precision={precision}", flush=True)
    wl = W.WORKLOADS["tiny"].with_(n_vpl=n_vpl, interleave=interleave, atlas_side=atlas, width=size[0], height=size[1],
                                   n_points=6_000, levels=2)
    inp = W.build_inputs(wl)
    rsm = mlgi.rsm_desc(ctx.upload(inp.rsm_diffuse), ctx.upload(inp.rsm_normal), ctx.upload(inp.rsm_depth), inp.inv_bvp)
    pts = mlgi.points_desc(ctx.upload(inp.points), ctx.upload(inp.bin_offsets))
    gb = mlgi.gbuffer_desc(ctx.upload(inp.gb_depth), ctx.upload(inp.gb_normal), inp.vp_inv)
    images = []
    for tile in ((8, 8), (16, 16), (32, 8), (16, 4)):
        p = wl.params(precision=precision)
        p.tile_w, p.tile_h = tile
        st = mlgi.GIStage(ctx, p, n_vpl, *size)
        st.process(rsm, pts, gb)
        ctx.sync()
        images.append(st.gi_buffer.numpy())
        b = mlgi.Batch(ctx, [(st, rsm, pts, gb)])
        b.run()
        ctx.sync()
        images.append(st.gi_buffer.numpy())
        b.close()
    for im in images[2::2]:
        assert np.array_equal(im, images[0])
    for im in images[3::2]:
        assert np.array_equal(im, images[1])
    rec, r16 = st.vpl_processor.host_records(), st.ism.pushpull_result.numpy()
    p = wl.params()
    ref, _ = oracle.final_gather(inp.gb_depth, inp.gb_normal, inp.vp_inv, rec[:, 0:3], rec[:, 4:7], rec[:, 16:19], r16,
                                 atlas, p.z_far, p.gi_intensity_factor, p.vpl_clamping_value, interleave)
    norm = np.linalg.norm(ref)
    for im in images[:2]:
        assert np.linalg.norm(im - ref) <= bar * norm


@pytest.mark.parametrize("shadowing", [True, False])
@pytest.mark.parametrize("size", [(33, 17), (256, 256), (260, 256), (352, 362), (362, 362)])
def test_record_fetch_forms(ctx, size, shadowing):
    """FP32: the next record requested ahead (launches of few waves; the sizes
    lie around 1,024 and 2,048 waves), each record requested in turn, and the
    batched kernel give the same bits."""
    print(f"[gather] fetch forms {size} shadowing={shadowing}", flush=True)
    wl = W.WORKLOADS["tiny"].with_(n_vpl=1024, interleave=2, atlas_side=512, width=size[0], height=size[1],
                                   n_points=6_000, levels=2)
    inp = W.build_inputs(wl)
    rsm = mlgi.rsm_desc(ctx.upload(inp.rsm_diffuse), ctx.upload(inp.rsm_normal), ctx.upload(inp.rsm_depth), inp.inv_bvp)
    pts = mlgi.points_desc(ctx.upload(inp.points), ctx.upload(inp.bin_offsets))
    gb = mlgi.gbuffer_desc(ctx.upload(inp.gb_depth), ctx.upload(inp.gb_normal), inp.vp_inv)
    images = []
    for fetch in (0, 1):
        p = wl.params(precision=mlgi.PRECISION_FP32)
        p.tile_w, p.tile_h, p.gather_fetch, p.enable_shadowing = 8, 8, fetch, int(shadowing)
        st = mlgi.GIStage(ctx, p, wl.n_vpl, *size)
        st.process(rsm, pts, gb)
        ctx.sync()
        images.append(st.gi_buffer.numpy())
    b = mlgi.Batch(ctx, [(st, rsm, pts, gb)])
    b.run()
    ctx.sync()
    images.append(st.gi_buffer.numpy())
    b.close()
    assert images[0].max() > 0
    assert np.array_equal(images[0], images[1]) and np.array_equal(images[0], images[2])
