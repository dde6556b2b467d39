"""Decode attention of one, two and four query heads per key/value head, whose keys and values go through the vector unit (csrc/hymix/
hm_attn_stream.h), against plain float64 attention: lengths around its steps of 32 keys, its tiles and its pairs of tiles, pages longer
than a tile, windows, kept first tokens, chunks, capped scores, sinks, and as many splits as leave some empty.  Rows of the cache that no
key of the step holds are NaN."""
import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nano-vllm-hw3_amd"))
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

from test_hymix_ops import batch, gen, rnd  # noqa: E402

from nanovllm import hy_ops  # noqa: E402

LENS = [1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 193, 257, 700]


def reference(q, k, v, n, scale, window, keep, chunk, cap, sink):
    """q [H, D], k and v [n, G, D] in float64 -> [H, D]."""
    H, G = q.shape[0], k.shape[1]
    k, v = (x.repeat_interleave(H // G, 1) for x in (k, v))
    s = (q[None] * k).sum(-1) * scale                                 # [n, H]
    if cap:
        s = cap * torch.tanh(s / cap)
    j, i = torch.arange(n)[:, None], n - 1
    seen = torch.ones(n, 1, dtype=torch.bool)
    if window:
        seen &= (i - j < window) | (j < keep)
    if chunk:
        seen &= j // chunk == i // chunk
    s = s.masked_fill(~seen, float("-inf"))
    if sink is not None:
        s = torch.cat([s, sink[None].double()])
    return (torch.softmax(s, 0)[:n, :, None] * v).sum(0)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,page", [(4, 4, 128, 64), (16, 8, 128, 64), (8, 2, 128, 192), (3, 3, 64, 128), (4, 2, 64, 64), (16, 4, 64, 64)])
@pytest.mark.parametrize("window,keep,chunk,cap,sink", [(0, 0, 0, 0.0, True), (0, 0, 0, 5.0, False), (64, 5, 0, 0.0, False), (33, 0, 0, 5.0, True),
                                                        (1, 70, 0, 0.0, True), (0, 0, 48, 0.0, False), (300, 0, 100, 0.0, True)])
def test_streamed_decode_attention(monkeypatch, H, G, D, page, window, keep, chunk, cap, sink):
    bf, scale = torch.bfloat16, 0.3
    g = gen(H + D + window + chunk)
    ctx, _ = batch([(n - 1, 1) for n in LENS], page, seed=H)
    rows = (int(ctx.block_tables.max()) + 1) * page
    kc, vc = (torch.full((rows, G, D), float("nan"), dtype=bf) for _ in range(2))
    q, sk = rnd(g, len(LENS), H, D, dtype=bf), rnd(g, H, s=2.0) if sink else None
    want, top = [], []
    for b, n in enumerate(LENS):
        at = ctx.block_tables[b].long()[torch.arange(n) // page] * page + torch.arange(n) % page
        kc[at], vc[at] = rnd(g, n, G, D, dtype=bf), rnd(g, n, G, D, dtype=bf)
        want.append(reference(q[b].double(), kc[at].double(), vc[at].double(), n, scale, window, keep, chunk, cap, sk))
        top.append(vc[at].double().abs().max())
    want, top = torch.stack(want), torch.stack(top)[:, None, None]
    ctx, _ = batch([(n - 1, 1) for n in LENS], page, device="cuda", seed=H)
    args = (q.cuda(), kc.view(-1, page, G, D).cuda(), vc.view(-1, page, G, D).cuda(), ctx, scale, sk.cuda() if sink else None, window, keep)
    for splits in (1, 3, 64):
        monkeypatch.setattr(hy_ops, "decode_splits", lambda *a: splits)
        got = hy_ops.paged_attention(*args, chunk=chunk, softcap=cap).view(want.shape).double().cpu()
        # one rounding to bf16 (2^-9 of the value), and weights whose scores carry the float32 error of D products and the exponential's
        # (scores to 40, 2e-6 of them at most) times the largest value
        assert (got - want).abs().le(2.0 ** -8 * want.abs() + 1e-4 * top).all()


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D", [(4, 2, 64), (16, 2, 128), (6, 2, 32)])            # (streamed; not)
@pytest.mark.parametrize("sink", [False, True])
def test_more_than_64_splits(monkeypatch, H, G, D, sink):
    """The merge beyond its 64 lanes: 130 tiles, which are 65 used splits of 65 or 130 where a split takes pairs of them, else 130."""
    bf, scale, page, lens = torch.bfloat16, 0.3, 64, [8320, 70, 8257]
    g = gen(H + D)
    ctx, _ = batch([(n - 1, 1) for n in lens], page, seed=H)
    rows = (int(ctx.block_tables.max()) + 1) * page
    kc, vc = (rnd(g, rows, G, D, dtype=bf) for _ in range(2))
    q, sk = rnd(g, len(lens), H, D, dtype=bf), rnd(g, H, s=2.0) if sink else None
    want = []
    for b, n in enumerate(lens):
        at = ctx.block_tables[b].long()[torch.arange(n) // page] * page + torch.arange(n) % page
        want.append(reference(q[b].double(), kc[at].double(), vc[at].double(), n, scale, 0, 0, 0, 0.0, sk))
    want, top = torch.stack(want), vc.double().abs().max()
    ctx, _ = batch([(n - 1, 1) for n in lens], page, device="cuda", seed=H)
    for splits in (64, 65, 130):
        monkeypatch.setattr(hy_ops, "decode_splits", lambda *a: splits)
        got = hy_ops.paged_attention(q.cuda(), kc.view(-1, page, G, D).cuda(), vc.view(-1, page, G, D).cuda(), ctx, scale,
                                     sk.cuda() if sink else None).view(want.shape).double().cpu()
        # a rounding to bf16; where the weights go through the matrix cores each is rounded too (2^-9 of it, so of the largest value at most)
        assert (got - want).abs().le(2.0 ** -8 * want.abs() + (1e-4 if D == 64 else 2.0 ** -9) * top).all(), splits
