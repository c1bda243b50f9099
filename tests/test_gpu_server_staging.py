"""GPU: served results on their way to the caller's memory. A batch whose
results do not all fit the server's pinned staging (three 1024^2 images against
16 MiB) delivers some through it and some directly; every image equals the one
served alone, also where requests leave theirs on the device, and a second
burst into the same arrays is delivered again."""
import numpy as np
import pytest

import mlgi
from mlgi import workloads as W

pytestmark = pytest.mark.gpu


def test_results_past_the_staging(ctx):
    srv = mlgi.Server(ctx, [(W._scene(1, 500), 20_000, 5)], [256], [(1024, 1024), (64, 48), (17, 9)],
                      hbm_budget=512 << 20, max_batch=6)
    sizes = [(1024, 1024), (64, 48), (1024, 1024), (17, 9), (1024, 1024), (64, 48), (17, 9), (1024, 1024)]

    def serve(spacing, seed, skip=()):
        reqs = [(0, w, h, 256, seed + k, k * spacing) for k, (w, h) in enumerate(sizes)]
        outs = [None if k in skip else np.full((h, w, 3), -1, np.float32) for k, (w, h) in enumerate(sizes)]
        st, _ = srv.run(reqs, outs)
        assert st["completed"] == len(reqs)
        return outs, st
    for seed in (10, 90):
        print(f"[serve] staging seed={seed}", flush=True)
        burst, st = serve(0.0, seed)
        assert st["mean_batch"] > 1.0
        alone, _ = serve(0.02, seed)
        some, _ = serve(0.0, seed, skip=(0, 3, 4))
        for k, (a, b, c) in enumerate(zip(burst, alone, some)):
            assert np.array_equal(a, b) and a.min() >= 0
            assert c is None or np.array_equal(c, b)
    srv.close()
