"""The expert tiles that a workgroup walks over (csrc/seqmix/sm_moe_tiles.hip) against the 32-row form, whose sums are the same bit for bit, where
the walk can go wrong: one tile and none for most workgroups, a last round by halves and by whole tiles, odd numbers of row tiles, tiles
of 128 and 256 rows, the fewest steps, outputs that end inside a tile, groups that end inside a block of 32 rows, weights on the input,
and one of the two products whose k is no multiple of 128.  And the gate: its quotient at the ends of its range, its special numbers."""
import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nano-vllm-hw3_amd"))

from nanovllm import seq_ops  # noqa: E402


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,E,W,F,act", [(1, 1, 1, 128, 128, "silu_glu"), (257, 1, 1, 128, 256, "silu_glu"), (300, 2, 3, 256, 136, "gelu"),
                                             (700, 2, 5, 384, 1152, "clamped_glu"), (513, 3, 4, 1152, 384, "relu_sq"),
                                             (4000, 2, 4, 256, 1536, "silu_glu"), (9001, 2, 3, 512, 1024, "clamped_glu"),
                                             (6000, 2, 7, 200, 2048, "silu_glu"), (8300, 1, 32, 2048, 264, "gelu"), (1000, 1, 1, 2048, 8192, "silu_glu")])
def test_walked_tiles_equal_the_small_ones(T, top, E, W, F, act):
    g = torch.Generator().manual_seed(T + W)
    parts = 2 if act.endswith("glu") else 1
    kind = dict(silu_glu=seq_ops.ACT_SILU_GLU, clamped_glu=seq_ops.ACT_CLAMPED_GLU, gelu=seq_ops.ACT_GELU, relu_sq=seq_ops.ACT_RELU_SQ)[act]
    h = torch.randn(T, W, generator=g).bfloat16().cuda()
    w_gu, w_down = ((torch.randn(E, *s, generator=g) * s[1] ** -0.5).bfloat16().cuda() for s in ((parts * F, W), (W, F)))
    # a last expert with few tokens, and the others as the numbers fall
    bent = torch.rand(T, E, generator=g) + torch.tensor([0.0] * (E - 1) + [-0.6 if E > top else 0.0])
    idx, wts = bent.topk(top, -1)[1].int().cuda(), torch.rand(T, top, generator=g).cuda()
    for weight_in in (False, True):
        a, b = (seq_ops.moe_experts(h, idx, wts, w_gu, w_down, 7.0, 1.702, form=f, act_kind=kind, weight_in=weight_in) for f in ("grouped", "tiles128"))
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)


@pytest.mark.gpu
def test_gate_at_the_ends_of_its_range():
    """g / (1 + e^-g) * u in float32: quotients by more than 2^126 and by infinity, subnormal gates, infinities."""
    g = torch.tensor([0.0, -0.0, 1e-30, 0.3, -0.3, 5.0, -5.0, 60.0, -60.0, -86.0, -87.3, -87.5, -88.0, -88.5, 2e38, 1e-40, -1e-40, -90.0, -200.0, -3e38,
                      float("inf")])                                                                                     # (1.5 g below 3.4e38)
    u = torch.full_like(g, 1.5)
    y = seq_ops.gated_act(torch.cat([g, u])[None].cuda(), seq_ops.ACT_SILU_GLU, float("inf"), 1.0)[0].cpu().double()
    want = g.double() / (1.0 + torch.exp(-g.double())) * 1.5
    # float32: the exponential's argument is rounded (2^-24 of up to 90) and the hardware's exponential is good to 2 units
    assert (y[:15] - want[:15]).abs().le(1.2e-5 * want[:15].abs()).all()
    assert (y[15:17] - want[15:17]).abs().le(2.9e-45).all()            # subnormal: two units, 2^-149 each
    assert (y[17:20] == 0).all()                                       # e^-g has left float32's range
    assert torch.isinf(y[20]) and y[20] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("act,alpha", [(seq_ops.ACT_SILU_GLU, 1.0), (seq_ops.ACT_CLAMPED_GLU, 1.702)])
@pytest.mark.parametrize("limit", [float("inf"), 7.0, 0.0, -3.0])
def test_gate_takes_minimum_and_maximum_as_the_library_does(dtype, act, alpha, limit):
    """Every pair of special numbers as gate and as up product: a NaN on either side, quiet or signalling, gives way to the limit (fmin, fmax), a
    negative limit is what both become, and what is then divided and multiplied follows the plain operations."""
    bits = torch.tensor([0x7fa00000, 0x7fc00000, -0x600000, 0x7f800000, -0x800000, 0, -0x80000000, 0x3f800000, -0x40800000, 0x41200000, -0x3ee00000,
                         0x7f7f0000, -0x810000], dtype=torch.int32)            # sNaN, qNaN, -sNaN, +-inf, +-0, +-1, +-10, +-the largest of bf16
    raw = torch.cat(torch.meshgrid(bits, bits, indexing="ij")).reshape(2, -1)
    x = raw.view(torch.float32) if dtype == torch.float32 else (raw >> 16).to(torch.int16).view(torch.bfloat16)
    y = seq_ops.gated_act(x.reshape(1, -1).cuda(), act, limit, alpha)[0].cpu()
    g, u = (torch.where(torch.isnan(v), torch.full_like(v, float("nan")), v) for v in x.double())
    top = torch.tensor(limit, dtype=torch.float64)
    g, u = torch.fmin(g, top), torch.fmin(torch.fmax(u, -top), top)
    want = (g / (1.0 + torch.exp(-alpha * g)) * (u + (0.0 if act == seq_ops.ACT_SILU_GLU else 1.0))).to(dtype)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    y, want = (torch.nan_to_num(v.double(), nan=0.0, posinf=1e300, neginf=-1e300) for v in (y, want))
    # the exponential's argument of up to 25 (base 2) and its factor are rounded (2^-20 and 2^-24 of it), and it has two units of its own; bf16: a rounding that falls the other way
    assert (y - want).abs().le((4e-6 if dtype == torch.float32 else 2.0 ** -7) * want.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,E", [(1, 1, 1), (16, 4, 3), (17, 4, 70), (1024, 4, 5), (1025, 4, 5), (4096, 1, 130), (4097, 1, 130), (63, 65, 200)])
def test_pairs_sorted_by_expert(T, top, E):
    """The grouping of pairs that a workgroup keeps in registers (up to 4096) and of more, by what the experts make of it: every one of
    them moves the columns by a number of its own (and beyond as many experts as columns doubles them), so that a pair which went to
    another would have its values elsewhere."""
    g = torch.Generator().manual_seed(T + E)
    W = F = 128
    idx = torch.randint(0, E, (T, top), generator=g).int()
    one, e = torch.eye(W), torch.arange(E)
    down = torch.stack([torch.roll(one, int(i) % W, 0) * 2.0 ** (int(i) // W) for i in e])
    w_gu, w_down = one.repeat(E, 1, 1).bfloat16(), down.bfloat16()
    h, wts = torch.randn(T, W, generator=g).abs().bfloat16(), torch.rand(T, top, generator=g)
    at = (torch.arange(W) - idx.long()[..., None] % W) % W
    want = (h.double() ** 2).bfloat16().double()[:, None].expand(T, top, W).gather(2, at) * (wts.double() * 2.0 ** (idx // W).double())[..., None]
    y = seq_ops.moe_experts(h.cuda(), idx.cuda(), wts.cuda(), w_gu.cuda(), w_down.cuda(), 7.0, form="grouped", act_kind=seq_ops.ACT_RELU_SQ).double().cpu()
    # the products are exact, the square is rounded to bf16 here as there (a tie may fall either way) and the sum once: 2^-8 of each
    assert (y - want.sum(1)).abs().le(2.0 ** -8 * want.sum(1) * 1.01 + 1e-30).all()
