"""The order in which the prompt attention kernels deal their row tiles (csrc/row_deal.h): on the CPU, the header itself compiled
with the host compiler; on the GPU, the time of a long prompt among single tokens."""
import ctypes
import os
import shutil
import subprocess

import pytest
import torch

from nanovllm import ops, seq_ops
from test_lilevik_ops import batch

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-hw3_amd", "csrc")
SOURCE = """#include "row_deal.h"
extern "C" void grid_of(int64_t tiles, int B, int G, uint32_t* out) {
    const RowGrid g = row_grid(tiles, B, G);
    out[0] = g.x; out[1] = g.y; out[2] = g.z; out[3] = (uint32_t)g.run;
}
extern "C" void walk(int tiles, int B, int G, int* seen, int* die) {     // [B][G][tiles]: how often, and on which die
    const RowGrid g = row_grid(tiles, B, G);
    uint64_t id = 0;
    for (uint32_t z = 0; z < g.z; ++z)
        for (uint32_t y = 0; y < g.y; ++y)
            for (uint32_t x = 0; x < g.x; ++x, ++id) {
                const RowTile t = row_tile(x, y, z, g.run, tiles, B, G);
                if (t.b < 0) continue;
                const uint64_t at = ((uint64_t)t.b * G + t.g) * tiles + t.tile;
                ++seen[at];
                die[at] = (int)(id & 7);
            }
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    where = tmp_path_factory.mktemp("row_deal")
    (where / "deal.cpp").write_text(SOURCE)
    subprocess.check_call([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(where / "deal.cpp"), "-o", str(where / "deal.so")])
    return ctypes.CDLL(str(where / "deal.so"))


@pytest.mark.parametrize("B,G", [(1, 1), (3, 2), (8, 1), (1, 8), (4, 2), (32, 1), (33, 1), (13, 3), (5, 8), (7, 16), (40, 6), (3, 24)])
@pytest.mark.parametrize("tiles", [1, 2, 7, 8, 9, 16, 63, 250])
def test_every_tile_once_and_a_sequence_on_every_die(deal, B, G, tiles):
    seen, die = torch.zeros(B, G, tiles, dtype=torch.int32), torch.zeros(B, G, tiles, dtype=torch.int32)
    deal.walk(tiles, B, G, ctypes.c_void_p(seen.data_ptr()), ctypes.c_void_p(die.data_ptr()))
    assert (seen == 1).all()
    pairs = B * G
    if pairs >= 32 or pairs % 8 == 0:
        # one sequence's tiles, all heads: no die has more than its eighth, in whole runs of eight tiles
        step = min(G & -G, 8)
        for b in range(B):
            load = torch.bincount(die[b].flatten().long(), minlength=8)
            assert load.max() <= -(-G // step) * 8 * -(-(-(-tiles // 8)) // (8 // step))
        # one tile alone, all that a single token has: spread over the dies too
        load = torch.bincount(die[:, :, 0].flatten().long(), minlength=8)
        assert load.max() - load.min() <= 1


@pytest.mark.parametrize("tiles,B,G", [(128, 20000, 8), (8192, 1024, 8), (2 ** 20, 64, 1), (2 ** 20 + 5, 8, 1), (1, 65535, 65535), (4096, 65535, 128)])
def test_grids_within_the_launch_limits(deal, tiles, B, G):
    """Fewer than 2^32 threads of 256 in x and at most 65535 groups in y and z, whatever number of sequences and heads is taken."""
    out = (ctypes.c_uint32 * 4)()
    deal.grid_of(ctypes.c_int64(tiles), B, G, out)
    assert out[0] * 256 < 2 ** 32 and out[1] <= 65535 and out[2] <= 65535
    assert out[0] * out[1] * out[2] >= tiles * B * G


def _us(f, n=20):
    for _ in range(5):
        f()
    best = float("inf")
    for _ in range(5):
        s, e = torch.cuda.Event(True), torch.cuda.Event(True)
        s.record()
        for _ in range(n):
            f()
        e.record()
        torch.cuda.synchronize()
        best = min(best, s.elapsed_time(e) / n * 1e3)
    return best


@pytest.mark.gpu
def test_one_prompt_among_single_tokens_has_the_whole_chip():
    """Latent attention of 2000 tokens beside 31 single ones of 900: little longer than the two of them apart, where all of the
    prompt's rows on one die took three times as long."""
    g = torch.Generator().manual_seed(1)

    def us(portions):
        ctx, blocks = batch(portions, device="cuda", seed=2)
        cache = torch.randn(blocks, 64, 256, generator=g).bfloat16().cuda()
        q = torch.randn(ctx.num_tokens, 16, 256, generator=g).bfloat16().cuda()
        return _us(lambda: seq_ops.latent_attention(q, cache, ctx, 0.06, value_cols=192))
    prompt, single = [(0, 2000)], [(899, 1)] * 31
    together, apart = us(prompt + single), us(prompt) + us(single)
    assert together <= 1.6 * apart, (together, apart)


@pytest.mark.gpu
def test_prompt_attention_of_more_pairs_than_one_grid_dimension_holds():
    """20000 sequences by 8 heads, the longest of 129 row tiles: more workgroups than 2^32 threads.  Every row is what it is in a call
    of its own sequence."""
    g = torch.Generator().manual_seed(3)
    lens = [16500] + [1] * 19999
    T = sum(lens)
    q, k, v = (torch.randn(T, 8, 128, generator=g).bfloat16().cuda() for _ in range(3))
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    out = ops.attn_prefill(q, k, v, cu, max(lens), 128 ** -0.5)
    n = lens[0]
    alone = ops.attn_prefill(q[:n], k[:n], v[:n], cu[:2], n, 128 ** -0.5)
    assert torch.equal(out[:n], alone)
    assert torch.equal(out[n:], v[n:])                     # a sequence of one token returns its value
