"""GPU: served results on their way to the caller's memory. A batch whose
results do not all fit the server's pinned staging (three 1024^2 images against
16 MiB) delivers some through it and some directly; every image equals the one
served alone, also where requests leave theirs on the device, and a second
burst into the same arrays is delivered again."""
import ctypes as C

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


def test_results_that_share_memory_or_are_pinned(ctx):
    """One array taken by all requests of a size holds one of their images
    whole, the last of its batch; pinned arrays are filled like others."""
    srv = mlgi.Server(ctx, [(W._scene(1, 500), 20_000, 5)], [256], [(512, 300), (64, 48)],
                      hbm_budget=256 << 20, max_batch=8, streams=1)
    reqs = [(0, 512, 300, 256, 20 + k, 0.0) for k in range(4)]
    own = [np.full((300, 512, 3), -1, np.float32) for _ in reqs]
    print("[serve] own arrays", flush=True)
    srv.run(reqs, own)
    shared = np.full((300, 512, 3), -1, np.float32)
    print("[serve] one array", flush=True)
    srv.run(reqs, [shared] * 4)
    assert np.array_equal(shared, own[3])
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library has loaded
    mem = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(mem), C.c_size_t(4 * own[0].nbytes), C.c_uint(0)) == 0
    pinned = np.frombuffer((C.c_char * (4 * own[0].nbytes)).from_address(mem.value), np.float32)
    pinned = pinned.reshape(4, 300, 512, 3)
    pinned[:] = -1
    print("[serve] pinned arrays", flush=True)
    srv.run(reqs, list(pinned))
    assert np.array_equal(pinned, np.stack(own))
    srv.close()
    del pinned
    assert hip.hipHostFree(mem) == 0
