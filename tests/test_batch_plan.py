"""What a batch's plan tells its launches (CPU only, no device): the tile pass
streams its stores from 176 MiB of tiles on, counted over the frames' own
atlases, whatever the largest ISM side among them; a server's staging slots
start on 256-byte lines for every number of slots; and the pull-push takes the
groups of ISMs that test_gpu_pullpush_groups.py means to run."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

import mlgi
from test_gpu_pullpush_groups import BATCHES, SINGLE

SRC = Path(__file__).with_name("batch_plan.cpp")
MIB = 1 << 20


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("plan") / "libplan.so"
    native = Path(mlgi.__file__).parent
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(SRC), "-o", str(so), f"-L{native}", "-l:libmlgi.so", f"-Wl,-rpath,{native}"], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("frames,mib,stream", [
    ([(4096, 4096)] + [(1024, 1024)] * 8, 96, False),  # ISMs of 64^2 beside 32^2
    ([(256, 1024)] + [(4096, 1024)] * 30, 124, False),  # of 64^2 beside 16^2
    ([(4096, 4096)] * 2 + [(4096, 2048)] * 3, 176, True),
    ([(1024, 1024)] * 43, 172, False),
    ([(1024, 1024)] * 44, 176, True),
])
def test_tile_bytes(lib, frames, mib, stream):
    n = len(frames)
    vpl, side = ((C.c_int * n)(*c) for c in zip(*frames))
    total, largest = C.c_uint64(0), C.c_int(0)
    assert lib.plan_tiles(n, vpl, side, C.byref(total), C.byref(largest)) == 0
    assert total.value == mib * MIB
    assert bool(lib.streams(total)) == stream


def test_stage_slots_are_aligned(lib):
    lib.stage_slot.argtypes, lib.stage_slot.restype = [C.c_int, C.c_size_t, C.c_int], C.c_size_t
    for slots in range(1, 65):
        for largest in (17 * 9 * 12, 1917 * 1079 * 12, 16384 * 16384 * 12):
            for batch in (1, 7, 32):
                b = lib.stage_slot(slots, largest, batch)
                assert b % 256 == 0 and b * slots <= 96 * MIB and b <= 16 * MIB
                assert b >= min(largest * batch, 16 * MIB, 96 * MIB // slots - 255)


def test_pullpush_groups(lib):
    assert {g for *_, g in SINGLE} == {4, 16, 64} == {g for *_, g in BATCHES}
    for side, n1d, group in SINGLE:
        assert lib.pp_group(side, n1d * n1d, 1) == group
    for side, n1d, frames, group in BATCHES:
        assert lib.pp_group(side, n1d * n1d, frames) == group
