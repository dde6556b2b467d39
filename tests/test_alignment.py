"""Operands that start on no 16-byte boundary (a contiguous view into a larger buffer): what is loaded straight to LDS elsewhere goes
through registers, with the same results."""
import pytest
import torch

from nanovllm import hy_ops, ops, seq_ops
from test_hymix_ops import batch, gen, near, rnd

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def off(t, by):
    """A contiguous copy of t that starts ``by`` elements behind a 16-byte boundary."""
    buf = torch.zeros(t.numel() + 8, dtype=t.dtype, device=t.device)
    view = buf[by:by + t.numel()].view(t.shape)
    view.copy_(t)
    assert view.is_contiguous() and (view.data_ptr() - by * t.element_size()) % 16 == 0
    return view


@pytest.mark.parametrize("by", [1, 4])
@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (4, 2), (8, 2)])
def test_prompt_attention(by, Hq, Hkv):
    g = gen(by + Hq)
    lens = [1, 65, 200, 64]
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    q, k, v = (rnd(g, sum(lens), h, 128).cuda().to(BF16) for h in (Hq, Hkv, Hkv))
    ref = ops.attn_prefill(q, k, v, cu, max(lens), 128 ** -0.5)
    for a, b in ((off(k, by), v), (k, off(v, by)), (off(k, by), off(v, by))):
        assert torch.equal(ops.attn_prefill(q, a, b, cu, max(lens), 128 ** -0.5), ref)


@pytest.mark.parametrize("by", [1, 4])
def test_paged_and_latent_attention(by):
    """Against the portable kernels (two bf16 roundings of values near one), prompts and single tokens."""
    g = gen(by)
    for portions in ([(0, 100), (130, 70), (0, 1), (64, 65)], [(99, 1), (64, 1), (300, 1)]):
        ctx, blocks = batch(portions, device="cuda", seed=by)
        q = rnd(g, ctx.num_tokens, 4, 128, s=0.7).cuda().to(BF16)
        kc, vc = (rnd(g, blocks, 64, 2, 128, s=0.7).cuda().to(BF16) for _ in range(2))
        kp, vp = (rnd(g, blocks, 4, 2, 128).cuda().to(BF16) for _ in range(2))
        for kw in (dict(), dict(window=40, pooled=(off(kp, by), vp, 16)), dict(window=40, pooled=(kp, off(vp, by), 16))):
            for a, b in ((off(kc, by), vc), (kc, off(vc, by)), (kc, vc)):
                near(hy_ops.paged_attention(q, a, b, ctx, 0.2, **kw),
                     hy_ops.paged_attention(q, kc, vc, ctx, 0.2, force_rows=True, **kw).double().cpu(), BF16, bf16=2e-2)
        ql, cache = rnd(g, ctx.num_tokens, 16, 256, s=0.7).cuda().to(BF16), rnd(g, blocks, 64, 256, s=0.7).cuda().to(BF16)
        near(seq_ops.latent_attention(ql, off(cache, by), ctx, 0.2, value_cols=192),
             seq_ops.latent_attention(ql, cache, ctx, 0.2, value_cols=192, force_rows=True).double().cpu(), BF16, bf16=2e-2)


@pytest.mark.parametrize("by", [1, 4])
@pytest.mark.parametrize("T,W,F,E,top", [(300, 200, 136, 3, 2), (900, 64, 264, 2, 1)])
def test_experts(by, T, W, F, E, top):
    """Tokens and tiled weights; 200 pairs per expert take tiles of 256 rows on boundaries, of 128 off them."""
    g = gen(T + by)
    h, idx = rnd(g, T, W).cuda().to(BF16), torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).int().cuda()
    w_gu, w_down = rnd(g, E, 2 * F, W, s=W ** -0.5).cuda().to(BF16), rnd(g, E, W, F, s=F ** -0.5).cuda().to(BF16)
    wts = torch.rand(T, top, generator=g).cuda()
    tiled = seq_ops.tile_expert_weights(w_gu, 2), seq_ops.tile_expert_weights(w_down)
    ref = seq_ops.moe_experts(h, idx, wts, w_gu, w_down, 1.2, form="tiles128", tiled=tiled)
    for x, t in ((off(h, by), tiled), (h, (off(tiled[0], by), tiled[1])), (h, (tiled[0], off(tiled[1], by)))):
        assert torch.equal(seq_ops.moe_experts(x, idx, wts, w_gu, w_down, 1.2, form="tiles128", tiled=t), ref)
