"""GPU: pull-push workgroups that take 4, 16 and 64 ISMs, which launches do that
still fill the chip with them (pullpush_group), against the oracle bit for bit:
groups without a sample (whose levels are not built), full ones and half empty
ones side by side, alone and in batches. That the library's rule gives these
groups for these sizes is checked on the CPU (test_batch_plan.py)."""
import numpy as np
import pytest

import mlgi
import oracle
from mlgi import workloads as W

pytestmark = pytest.mark.gpu

# ISM side, ISMs per atlas side, ISMs per workgroup
SINGLE = [(8, 64, 4), (8, 128, 16), (8, 256, 64), (16, 64, 4), (16, 128, 16), (32, 64, 4)]
# ISM side, ISMs per atlas side, frames, ISMs per workgroup
BATCHES = [(8, 128, 4, 64), (16, 64, 4, 16), (32, 32, 4, 4)]


def group_atlas(ism_side, n1d, group, seed):
    rng = np.random.default_rng(seed)
    side, n = n1d * ism_side, n1d * n1d
    kind = rng.integers(0, 3, n // group)  # empty, full, half empty
    kind[:3] = (0, 1, 2)
    density = np.repeat(np.array([0.0, 0.3, 0.3])[kind], group)
    density[np.repeat(kind == 2, group) & (np.arange(n) % group >= group // 2)] = 0.0
    p_full = np.repeat(np.repeat(density.reshape(n1d, n1d), ism_side, 0), ism_side, 1)
    texel = rng.integers(1 << 26, 1 << 32, (side, side), dtype=np.uint32)
    return np.where(rng.random((side, side), np.float32) < p_full, texel, np.uint32(0xFFFFFFFF)).astype(np.uint32)


@pytest.mark.parametrize("ism_side,n1d,group", SINGLE)
def test_groups(ctx, ism_side, n1d, group):
    side = n1d * ism_side
    atlas = group_atlas(ism_side, n1d, group, n1d + ism_side)
    for levels in sorted({1, 2, int(np.log2(ism_side))}):
        print(f"[pullpush] S={ism_side} L={levels} atlas={side} group={group}", flush=True)
        ism = mlgi.ImperfectShadowmap(ctx, side, n1d * n1d)
        assert ism.ism_side == ism_side
        ism.softrender.copy_from(atlas)
        ism.pushpull_result.copy_from(np.zeros((side, side), np.uint16))
        ism.pullpush(mlgi.default_params(atlas_side=side, z_far=50.0, pull_push_levels=levels))
        ctx.sync()
        assert np.array_equal(ism.pushpull_result.numpy(), oracle.pullpush(atlas, ism_side, levels, 50.0, threads=8))


@pytest.mark.parametrize("ism_side,n1d,frames,group", BATCHES)
def test_groups_in_batches(ctx, ism_side, n1d, frames, group):
    print(f"[pullpush] batch S={ism_side} n1d={n1d} x {frames} group={group}", flush=True)
    wl = W.WORKLOADS["tiny"].with_(n_vpl=n1d * n1d, interleave=4, atlas_side=n1d * ism_side, n_points=4 * n1d * n1d,
                                   levels=2)
    inp = W.build_inputs(wl)
    rsm = mlgi.rsm_desc(ctx.upload(inp.rsm_diffuse), ctx.upload(inp.rsm_normal), ctx.upload(inp.rsm_depth), inp.inv_bvp)
    gb = mlgi.gbuffer_desc(ctx.upload(inp.gb_depth), ctx.upload(inp.gb_normal), inp.vp_inv)
    stages, descs = [mlgi.GIStage(ctx, wl.params(), wl.n_vpl, wl.width, wl.height) for _ in range(frames)], []
    rng = np.random.default_rng(7)
    bins = np.repeat(np.arange(wl.n_vpl), np.diff(inp.bin_offsets))
    for st in stages:  # runs of 256 bins without a point leave whole groups empty and others in part
        full = np.append([False, True], rng.random(wl.n_vpl // 256 - 2) < 0.5)
        keep = full[bins // 256]
        off = np.append(0, np.cumsum(np.bincount(bins[keep], minlength=wl.n_vpl))).astype(np.uint32)
        descs.append((st, rsm, mlgi.points_desc(ctx.upload(inp.points[keep]), ctx.upload(off)), gb))
    b = mlgi.Batch(ctx, descs)
    b.run()
    ctx.sync()
    for st in stages:
        atlas = st.ism.softrender.numpy()
        isms = (atlas != 0xFFFFFFFF).reshape(n1d, ism_side, n1d, ism_side).any((1, 3)).reshape(-1, group)
        assert not isms.any(1).all() and isms.all(1).any()
        assert np.array_equal(st.ism.pushpull_result.numpy(),
                              oracle.pullpush(atlas, ism_side, wl.levels, st.params.z_far, threads=8))
    b.close()
