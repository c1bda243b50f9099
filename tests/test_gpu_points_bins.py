"""GPU: places of device-sampled points, counted in LDS up to 4,096 bins of at
least 64 points on average and in memory otherwise: offsets and every bin's
records equal the host sampler's at the edges of the workgroups' runs (1,024
points, 512 workgroups), of the 64 bins a scan workgroup takes, of the 2,048
runs of triangles the search starts with, and of the rule."""
import numpy as np
import pytest

import mlgi
from mlgi import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_points,n_bins,n_random", [(1, 1, 500), (64, 1, 500), (1023, 15, 500),
                                                      (1025, 16, 2036), (5_000, 65, 2037),
                                                      (524_289, 256, 4_000), (1_100_003, 4096, 40_000),
                                                      (262_143, 4096, 500), (262_144, 4096, 500),
                                                      (300_000, 4097, 500)])
def test_places_equal_host(ctx, n_points, n_bins, n_random):
    print(f"[points] n={n_points} bins={n_bins} tris={n_random + 12}", flush=True)
    scene = W._scene(1, n_random)
    dev = scene.upload(ctx)
    rec_h, off_h = scene.sample_points(n_points, n_bins, n_bins, 3)
    rec_d, off_d = dev.sample_points(n_points, n_bins, n_bins, 3)
    off = off_d.numpy()
    assert np.array_equal(off, off_h)
    bins = np.repeat(np.arange(n_bins), np.diff(off.astype(np.int64)))
    a, b = (np.ascontiguousarray(r[:n_points]).view(np.uint32) for r in (rec_d.numpy(), rec_h))
    for r in (a, b):
        r[:] = r[np.lexsort((*r.T, bins))]
    assert np.array_equal(a, b)
    dev.close()
