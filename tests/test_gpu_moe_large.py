"""Routing (on the matrix cores for many tokens, a workgroup per token for few) and the grouping by several workgroups."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-hw3_amd"))
from nanovllm import seq_ops  # noqa: E402

pytestmark = pytest.mark.gpu


def gen(seed):
    return torch.Generator().manual_seed(seed)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,E,top,groups,keep,gate", [
    (2048, 32, 16, 4, 1, 1, False), (2049, 544, 15, 3, 1, 1, True), (2063, 1024, 16, 2, 1, 1, True), (2050, 2048, 32, 4, 4, 2, False),
    (2101, 1056, 33, 5, 1, 1, False), (2048, 4096, 64, 8, 8, 3, False), (2055, 1568, 63, 1, 1, 1, True), (2047, 96, 1, 1, 1, 1, False),
    (1, 4100, 17, 4, 1, 1, True), (300, 1028, 16, 2, 1, 1, False), (77, 2052, 6, 2, 3, 2, True), (1023, 4, 5, 1, 1, 1, False)])
def test_route(dtype, T, W, E, top, groups, keep, gate):
    """Against 64-bit logits.  The sum of W products in float32 is off by at most W 2^-24 of the sum of their sizes (about sqrt(2 W / pi)
    times the spread of a logit, which is 1): below 4096 * 2^-24 * 51 = 0.013 at worst, some sqrt(W) 2^-24 = 4e-6 in fact.  So a chosen
    score lies within 1e-4 of the one the reference chooses in its place, and the weights likewise."""
    g = gen(T + E)
    h = torch.randn(T, W, generator=g).to(dtype)
    rw = torch.randn(E, W, generator=g) * W ** -0.5
    gw = torch.randn(W, generator=g) * W ** -0.5
    res = seq_ops.moe_route(h.cuda(), rw.cuda(), top, groups, keep, gate_w=gw.cuda() if gate else None)
    idx, wts = res[0].cpu().long(), res[1].cpu().double()
    p = torch.softmax(h.double() @ rw.double().t(), -1)
    c = p.clone()
    if groups > 1:
        best = c.view(T, groups, -1).amax(-1)
        kept = best.topk(keep, -1).indices
        near = best.sort(-1, descending=True).values
        sure = near[:, keep - 1] - near[:, keep] > 1e-5                   # rows whose kept groups do not hang on a rounding
        drop = torch.ones(T, groups, dtype=torch.bool).scatter(1, kept, False)
        c = c.masked_fill(drop.repeat_interleave(E // groups, 1), -1.0)
    else:
        sure = torch.ones(T, dtype=torch.bool)
    assert sure.float().mean() > 0.95
    ref = c.topk(top, -1).values
    got = c.gather(1, idx)
    assert (got - ref).abs()[sure].max() < 1e-4
    assert all(len(set(r)) == top for r in idx[:: 97].tolist())
    w = ref / ref.sum(-1, keepdim=True)
    assert (wts - w).abs()[sure].max() < 1e-4
    if gate:
        assert (res[2].cpu().double() - torch.sigmoid(h.double() @ gw.double())).abs().max() < 1e-4


@pytest.mark.parametrize("T,top,E,skew", [(6144, 2, 5, 0), (12288, 1, 3, 1), (12287, 1, 8, 0), (4099, 3, 70, 0), (3073, 4, 1000, 0), (70001, 2, 16, 2)])
def test_grouping_of_many_pairs(T, top, E, skew):
    """The large tiles' grouping (several workgroups from 12288 pairs on) against the small tiles' (one): the same bits, since a row's
    sums do not depend on the tile it sits in.  skew 1: all pairs to one expert; 2: most of them, and the last expert without any."""
    W, F = 64, 16
    g = gen(T)
    h = torch.randn(T, W, generator=g).cuda().bfloat16()
    score = torch.rand(T, E, generator=g)
    if skew:
        score[:, 0] += 2.0
        score[:, -1] -= 2.0
    idx = score.topk(top, -1).indices.int().cuda()
    wts = torch.rand(T, top, generator=g).cuda()
    w_gu = (torch.randn(E, 2 * F, W, generator=g) * W ** -0.5).cuda().bfloat16()
    w_down = (torch.randn(E, W, F, generator=g) * F ** -0.5).cuda().bfloat16()
    a, b = (seq_ops.moe_experts(h, idx, wts, w_gu, w_down, 7.0, form=f) for f in ("grouped", "tiles128"))
    assert torch.equal(a, b)
