"""Prompt attention by tiles against the form that goes row by row: tiles with keys behind a row's own, in front of its window or chunk, both, kept
first tokens and pooled blocks, with and without a cap, in the head sizes whose tiles go straight to LDS and in others; and the two forms by
tiles against each other, which do the same arithmetic."""
import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nano-vllm-hw3_amd"))
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

from test_hymix_ops import batch, gen, rnd  # noqa: E402

from nanovllm import hy_ops  # noqa: E402

BF = torch.bfloat16


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V", [(2, 1, 32, 32), (4, 4, 64, 64), (4, 2, 128, 128), (2, 2, 128, 64), (2, 1, 72, 40)])
@pytest.mark.parametrize("cap", [0.0, 1.5, 50.0])
@pytest.mark.parametrize("kind", ["plain", "window", "narrow", "kept", "chunk", "pooled"])
def test_one_sided_masks(H, G, D, V, cap, kind):
    g = gen(H + D + V)
    ctx, _ = batch([(0, 333), (70, 200), (129, 1), (0, 64)], 64, device="cuda", seed=D)
    pages = int(ctx.block_tables.max()) + 1
    k, v, q = rnd(g, pages, 64, G, D, dtype=BF).cuda(), rnd(g, pages, 64, G, V, dtype=BF).cuda(), rnd(g, ctx.num_tokens, H, D, dtype=BF).cuda()
    sink = rnd(g, H).cuda()
    kw = {"plain": dict(sink=sink), "window": dict(window=100, sink=sink), "narrow": dict(window=1), "kept": dict(window=65, keep_first=67),
          "chunk": dict(chunk=48), "pooled": dict(window=40)}[kind]
    if kind == "pooled":
        rows = hy_ops.pool_rows_per_page(64, 16)
        kp, vp = (torch.zeros(pages, rows, G, n, dtype=BF, device="cuda") for n in (D, V))
        whole, _ = batch([(0, 333), (0, 270), (0, 130), (0, 64)], 64, device="cuda", seed=D)
        hy_ops.pool_blocks(k, v, kp, vp, 16, whole)
        kw["pooled"] = (kp, vp, 16)
    got, want = (hy_ops.paged_attention(q, k, v, ctx, 2.0 * D ** -0.5, softcap=cap, force_rows=rows, **kw).double() for rows in (False, True))
    # two roundings to bf16 (2^-8 of the value) and the weights' (2^-9 of the largest value)
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -9 * v.double().abs().max()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D,V,less", [(128, 128, 120), (64, 64, 56), (128, 64, 56)])
@pytest.mark.parametrize("cap", [0.0, 1.5, 50.0, 30000.0])
@pytest.mark.parametrize("kind", ["plain", "window", "kept", "chunk"])
def test_tiles_straight_to_lds_give_the_same_bits(D, V, less, cap, kind):
    """Heads of 32, 64 or 128 channels go to LDS as they are, others through registers, with scores, maxima and sums of the same order: a value
    column's results do not depend on how many there are."""
    g = gen(D + V)
    ctx, _ = batch([(0, 333), (70, 200), (129, 1), (0, 64)], 64, device="cuda", seed=D)
    pages, H, G, T = int(ctx.block_tables.max()) + 1, 4, 2, ctx.num_tokens
    k, v, q = rnd(g, pages, 64, G, D, dtype=BF).cuda(), rnd(g, pages, 64, G, V, dtype=BF).cuda(), rnd(g, T, H, D, dtype=BF).cuda()
    kw = {"plain": dict(sink=rnd(g, H).cuda()), "window": dict(window=100), "kept": dict(window=65, keep_first=67), "chunk": dict(chunk=48)}[kind]
    slim, wide = (hy_ops.paged_attention(q, k, x.contiguous(), ctx, 2.0 * D ** -0.5, softcap=cap, **kw).view(T, H, -1) for x in (v, v[..., :less]))
    assert torch.equal(slim[..., :less], wide)
