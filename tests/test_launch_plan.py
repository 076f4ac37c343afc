"""Grids that grow with the largest inputs stay within what a launch takes."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vrad_amd", "csrc")
SRC = """
#include "launch_plan.h"
extern "C" {
int64_t grid_part(int64_t at, int64_t n, int t) { return vr::grid_part(at, n, t); }
int block_fill_slots(int64_t b) { return vr::block_fill_slots(b); }
int64_t block_fill_groups(int64_t b) { return vr::block_fill_groups(b); }
int64_t pair_launch_groups(int64_t p, int c) { return vr::pair_launch_groups(p, c); }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SRC)
    so = str(d / "plan.so")
    subprocess.run(["g++", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, "-o", so,
                    str(d / "plan.cpp")], check=True)
    lib = C.CDLL(so)
    for f in (lib.grid_part, lib.block_fill_slots, lib.block_fill_groups):
        f.restype = C.c_int64
    lib.pair_launch_groups.restype = C.c_int64
    lib.pair_launch_groups.argtypes = [C.c_int64, C.c_int]
    lib.grid_part.argtypes = [C.c_int64, C.c_int64, C.c_int]
    lib.block_fill_slots.argtypes = lib.block_fill_groups.argtypes = [C.c_int64]
    return lib


def parts(plan, groups, threads):
    at, out = 0, []
    while at < groups:
        out.append(plan.grid_part(at, groups, threads))
        assert out[-1] > 0 and out[-1] * threads < 2 ** 32
        at += out[-1]
    assert at == groups
    return out


# rows up to the most a batched or served set may have (2048^2), tiles of 2048
# and 4096 columns (at most 1024 of them)
@pytest.mark.parametrize("cols", [2048, 4096])
@pytest.mark.parametrize("rows", [1, 5970, 262144, 1840000, 2 ** 21, 3000000, 2048 ** 2])
def test_blocked_copy_launches(plan, rows, cols):
    tiles = -(-rows // cols)
    if tiles > 1024:
        return
    chunks = min(256, -(-rows // 256)) if rows <= 2 ** 18 else 256 * -(-rows // 2 ** 18)
    blocks = chunks * tiles
    slots = plan.block_fill_slots(blocks)
    assert plan.block_fill_groups(blocks) * 4 * slots >= blocks * 1024  # every slot has a wave
    fill = parts(plan, plan.block_fill_groups(blocks), 256)
    assert len(fill) == 1 or rows > 2 ** 20  # ordinary sets: one launch
    parts(plan, blocks, 1024)  # the offsets' launch, a workgroup per block


@pytest.mark.parametrize("chunk", [256, 1024, 8192])
@pytest.mark.parametrize("batch", [-1, 0, 1, 5000, 50000, 32 << 20, 2 ** 31 - 1])
def test_pair_launch_is_bounded(plan, batch, chunk):
    """A launch of MakeTransfers' trace holds batch_pairs candidate pairs at
    most, or one workgroup's run of them; in any case it fits a launch."""
    groups = plan.pair_launch_groups(batch, chunk)
    assert groups >= 1 and groups * 64 < 2 ** 32
    if batch > 0:
        assert groups == 1 or groups * chunk <= batch
