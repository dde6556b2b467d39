"""How the 32-row form of the experts deals its workgroups (csrc/seqmix/sm_moe_deal.h), on the CPU: the header itself compiled with the host
compiler."""
import ctypes
import os
import shutil
import subprocess

import pytest
import torch

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-hw3_amd", "csrc", "seqmix")
SOURCE = """#include "sm_moe_deal.h"
extern "C" void grid_of(int tiles, int columns, uint32_t* out) {
    const MoeGrid g = moe_grid(tiles, columns);
    out[0] = g.x; out[1] = g.y; out[2] = g.z;
}
// [tiles][blocks of 32 columns]: how often, on which die, and which workgroup of the die; out: workgroups with nothing to do
extern "C" long long walk(int tiles, int columns, int* seen, int* on, int* turn) {
    const MoeGrid g = moe_grid(tiles, columns);
    const int blocks = (columns + 31) / 32;
    uint64_t id = 0;
    long long idle = 0;
    for (uint32_t z = 0; z < g.z; ++z)
        for (uint32_t y = 0; y < g.y; ++y)
            for (uint32_t x = 0; x < g.x; ++x, ++id) {
                const MoePlace p = moe_place(x, y, z);
                if (p.block >= blocks || p.tile >= tiles) { ++idle; continue; }
                const uint64_t at = (uint64_t)p.tile * blocks + p.block;
                ++seen[at];
                on[at] = (int)(id & 7);
                turn[at] = (int)(id >> 3);
            }
    return idle;
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    where = tmp_path_factory.mktemp("moe_deal")
    (where / "deal.cpp").write_text(SOURCE)
    subprocess.check_call([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(where / "deal.cpp"), "-o", str(where / "deal.so")])
    return ctypes.CDLL(str(where / "deal.so"))


@pytest.mark.parametrize("tiles,columns", [(t, c) for t in (1, 7, 10, 13, 33) for c in (8, 32, 40, 248, 256, 264, 768, 1000, 1536, 2048)] +
                                          [(t, c) for t in (32768, 32770) for c in (8, 256)])
def test_every_block_of_every_tile_once_and_evenly(deal, tiles, columns):
    seen, on, turn = (torch.zeros(tiles, (columns + 31) // 32, dtype=torch.int32) for _ in range(3))
    deal.walk(tiles, columns, *(ctypes.c_void_p(t.data_ptr()) for t in (seen, on, turn)))
    assert (seen == 1).all()
    blocks = on.shape[1]
    assert (on == torch.arange(blocks) % 8).all()                  # a block's tiles on one die
    # the used tiles are the first ones: of their workgroups no CU of a die has more than its share, rounded up
    if columns % 256 == 0:
        for used in {1, tiles // 3, tiles * 2 // 3, tiles} - {0}:
            cu = (on[:used] * 32 + turn[:used] % 32).flatten().long()
            assert torch.bincount(cu, minlength=256).max() <= -(-used * (blocks // 8) // 32)


@pytest.mark.parametrize("columns", [8, 2048, 2 ** 20])
@pytest.mark.parametrize("pairs", [2 ** 20, 2 ** 25, 2 ** 28, 2 ** 30])
def test_grids_within_the_launch_limits(deal, pairs, columns):
    """Fewer than 2^32 threads of 64 in x and at most 65535 groups in y and z, up to the most pairs and experts that are taken."""
    tiles = pairs // 32 + 4096
    out = (ctypes.c_uint32 * 3)()
    deal.grid_of(tiles, columns, out)
    assert out[0] * 64 < 2 ** 32 and out[1] <= 65535 and out[2] <= 65535 and out[1] * out[2] >= tiles and out[0] * 32 >= columns
