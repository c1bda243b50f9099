"""Pull-push of ISMs without a sample. The device writes 65535 for a group of
ISMs whose tiles are all empty without building their levels: on the CPU, the
oracle's full pull-push gives 65535 in every texel for every ISM side, level
count and far plane; on the GPU, atlases whose groups are empty, full and half
empty side by side equal the oracle's bit for bit."""
import numpy as np
import pytest

import mlgi
import oracle

CASES = [(s, l) for s in (8, 16, 32, 64) for l in range(1, int(np.log2(s)) + 1)]


@pytest.mark.parametrize("ism_side,levels", CASES)
def test_empty_isms_are_far(ism_side, levels):
    atlas = np.full((ism_side, ism_side), 0xFFFFFFFF, np.uint32)
    for z_far in [2.0 ** k for k in range(-60, 61, 5)] + [0.05, 50.0, 33.3]:
        assert (oracle.pullpush(atlas, ism_side, levels, np.float32(z_far)) == 65535).all(), z_far


@pytest.mark.gpu
@pytest.mark.parametrize("ism_side,levels", CASES)
def test_empty_groups(ctx, ism_side, levels):
    side = max(256, 4 * ism_side)
    print(f"[pullpush] empty groups S={ism_side} L={levels}", flush=True)
    rng = np.random.default_rng(ism_side + levels)
    n1d = side // ism_side
    group = min((64 // ism_side) ** 2, n1d * n1d)  # ISMs in a row-major run of one workgroup
    kind = rng.integers(0, 3, n1d * n1d // group)
    kind[:3] = (0, 1, 2)
    density = np.repeat(np.array([0.0, 0.3, 0.3])[kind], group)
    density[np.repeat(kind == 2, group) & (np.arange(n1d * n1d) % group >= (group + 1) // 2)] = 0.0  # half empty
    p_full = np.repeat(np.repeat(density.reshape(n1d, n1d), ism_side, 0), ism_side, 1)
    texel = (rng.integers(1 << 18, 1 << 24, (side, side), dtype=np.uint32) << 8) | rng.integers(0, 256, (side, side),
                                                                                               dtype=np.uint32)
    atlas = np.where(rng.random((side, side)) < p_full, texel, np.uint32(0xFFFFFFFF)).astype(np.uint32)
    for z_far in (50.0, 2.0 ** -60, 2.0 ** 60):
        ism = mlgi.ImperfectShadowmap(ctx, side, n1d * n1d)
        assert ism.ism_side == ism_side
        ism.softrender.copy_from(atlas)
        ism.pushpull_result.copy_from(np.zeros((side, side), np.uint16))
        ism.pullpush(mlgi.default_params(atlas_side=side, z_far=z_far, pull_push_levels=levels))
        ctx.sync()
        assert np.array_equal(ism.pushpull_result.numpy(), oracle.pullpush(atlas, ism_side, levels, z_far))
