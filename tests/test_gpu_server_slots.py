"""GPU: a server whose seven staging slots share 96 MiB unevenly, and whose
odd-sized results follow one another in them: every image of a burst over all
slots equals the one served alone."""
import numpy as np
import pytest

import mlgi
from mlgi import workloads as W

pytestmark = pytest.mark.gpu


def test_seven_slots(ctx):
    sizes = [(512, 511), (17, 9), (63, 31)]
    srv = mlgi.Server(ctx, [(W._scene(1, 500), 20_000, 5)], [256], sizes, hbm_budget=512 << 20, max_batch=4,
                      max_queued_batches=7)
    reqs = [(0, *sizes[k % 3], 256, 40 + k, 0.0) for k in range(28)]

    def serve(requests):
        outs = [np.full((r[2], r[1], 3), -1, np.float32) for r in requests]
        st, _ = srv.run(requests, outs)
        assert st["completed"] == len(requests)
        return outs
    print("[serve] seven slots", flush=True)
    burst = serve(reqs)
    for r, got in zip(reqs, burst):
        alone, = serve([r])
        assert got.min() >= 0 and np.array_equal(got, alone)
    srv.close()
