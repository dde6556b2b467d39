"""Every mechanism the Kuporax family added to the operators, alone, against the plain restatement in
tests/oracle_kuporax.py: on the CPU the engine's plumbing operators, on the GPU (marked gpu) the HIP kernels of libhymix
and libseqmix in float32 and bfloat16.  Batches are built by hand: several sequences, portions that start in the middle
of a sequence, scattered cache blocks and state slots that hold stale data."""
import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nano-vllm-hw3_amd"))
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

import oracle_kuporax as O  # noqa: E402
from test_hymix_ops import CASES, F64, batch, gen, near, rnd  # noqa: E402  (operator test helpers)
from test_lilevik_ops import module, run_cut, stale  # noqa: E402

from nanovllm import hy_ops, seq_ops  # noqa: E402
from nanovllm.layers import gated_delta  # noqa: E402
from nanovllm.layers.gated_delta import GatedDelta  # noqa: E402
from nanovllm.layers.mixer_pair import MixerPair  # noqa: E402
from nanovllm.layers.rotary_attention import PagedRotaryAttention  # noqa: E402
from nanovllm.layers.state_space import StateSpaceDual  # noqa: E402

CUTS = [[37, 3, 1, 40, 1, 1, 7], [50], [2, 1, 1, 5]]
LENGTHS = [90, 50, 9]


# ------------------------------------------------------------------------------------------ residual side
@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("W,groups", [(40, 1), (7, 1), (264, 1), (1028, 1), (2600, 1), (4100, 1), (17000, 1), (3001, 1), (264, 4)])
def test_norms_around_sublayers(device, dtype, W, groups):
    """Embedding row plus position row (no norm) with the first norm; the boundary with both norms, weights stored around
    zero; the write alone; a residual far larger than what is added."""
    g = gen(W)
    T, eps = 9, 1e-4
    embed, table = rnd(g, 19, W, dtype=dtype), rnd(g, 30, W, s=0.5, dtype=dtype)
    ids, pos = torch.randint(0, 19, (T,), generator=g), torch.randperm(30, generator=g)[:T].int()
    w1, w2 = rnd(g, W, s=0.3, dtype=dtype), rnd(g, W, s=0.3, dtype=dtype)

    def norm(z, w, add):
        return O.rms(z.view(T, groups, -1), eps).view(T, W) * (add + w.to(F64))
    x, h = hy_ops.group_norm_residual(None, embed.to(device), None, groups, eps, dtype, next_w=w1.to(device), ids=ids.to(device), w_add=1.0,
                                      pos=pos.to(device), pos_table=table.to(device))
    ref = embed[ids].to(F64) + table[pos.long()].to(F64)
    near(x, ref, torch.float32, f32=1e-6)
    near(h, norm(ref, w1, 1), dtype)
    assert x.dtype == torch.float32 and h.dtype == dtype
    y = rnd(g, T, W, s=0.01, dtype=dtype)
    for add in (1.0, 0.0):
        x, h = hy_ops.group_norm_residual(x, y.to(device), w2.to(device), groups, eps, dtype, next_w=w1.to(device), w_add=add)
        ref = ref + norm(y.to(F64), w2, add)
        near(x, ref, torch.float32, f32=3e-6)
        near(h, norm(ref, w1, add), dtype)
    x, h = hy_ops.group_norm_residual(x, y.to(device), w2.to(device), groups, eps, dtype, want_h=False, w_add=1.0)
    near(x, ref + norm(y.to(F64), w2, 1), torch.float32, f32=3e-6)
    assert h is None
    x, h = hy_ops.group_norm_residual(None, embed.to(device), None, groups, eps, dtype, ids=ids.to(device))
    near(h, embed[ids].to(F64), dtype, f32=1e-6)


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("C,taps,start", [(40, 4, 24), (40, 4, 13), (7, 2, 3), (64, 1, 0), (1100, 3, 1096), (24, 5, 24), (16, 16, 8)])
def test_short_conv_with_silu_on_some_channels(device, dtype, C, taps, start):
    g = gen(C + taps)
    w, b = rnd(g, C, taps, s=0.6, dtype=dtype), rnd(g, C, s=0.5, dtype=dtype)
    hs = [rnd(g, n, 2 * C, dtype=dtype) for n in LENGTHS]
    refs = []
    for h in hs:
        r = O.causal_conv(h[:, C:].to(F64), w.to(F64), b.to(F64))
        r[:, start:] = O.silu(r[:, start:])
        refs.append(r)
    st = {}

    def caches(blocks, slots):
        st["s"] = torch.empty(slots, 1, max(taps - 1, 1), C, dtype=dtype, device=device)
        stale(st["s"], g)
    outs = run_cut(None, hs, CUTS, device, dtype, C, caches, forward=lambda x: seq_ops.short_conv(
        x[:, C:], w.to(device), st["s"], 0, seq_ops.get_step(), b.to(device), silu=True, silu_from=start))
    for o, r in zip(outs, refs):
        near(o, r, dtype)


# ------------------------------------------------------------------------------------------ recurrences
OUTER_SIZES = [(1, 1, 1, 1), (4, 2, 16, 24), (3, 3, 33, 7), (6, 2, 64, 40), (2, 1, 128, 72), (2, 2, 136, 16), (2, 1, 256, 130), (8, 1, 8, 8)]


def forget(g, H):
    """Decay rates from hardly any to nearly all per unit step, and biases that spread the steps."""
    return -torch.exp(rnd(g, H, s=1.5)), rnd(g, H) - 1.0


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("H,G,D,V", OUTER_SIZES)
def test_gated_delta_operator(device, dtype, H, G, D, V):
    """The recurrence alone: portions and single tokens (different kernels), heads that share keys, sizes on and off the
    register tiles, rows and pre-activations that are column slices, slots full of another sequence's state."""
    g = gen(H * 7 + D)
    A, bias = forget(g, H)
    n_qk = 2 * G * D
    hs = [torch.cat([rnd(g, n, n_qk, dtype=dtype), rnd(g, n, H * V, dtype=dtype), rnd(g, n, 2 * H, s=2.0, dtype=dtype)], 1) for n in LENGTHS]
    refs, of = [], torch.arange(H) // (H // G)
    for h in hs:
        h = h.to(F64)
        n = h.shape[0]
        q, k = O.unit(h[:, :G * D].reshape(n, G, D)) * 0.37, O.unit(h[:, G * D:n_qk].reshape(n, G, D))
        b, a = h[:, n_qk + H * V:].split([H, H], 1)
        refs.append(O.gated_delta(q[:, of], k[:, of], h[:, n_qk:n_qk + H * V].reshape(n, H, V), torch.sigmoid(b),
                                  torch.exp(A.to(F64) * O.softplus(a + bias.to(F64))))[0].reshape(n, H * V))
    st = {}

    def caches(blocks, slots):
        st["s"] = torch.empty(slots, H, D, V, device=device)
        stale(st["s"], g)

    def step(x):
        return hy_ops.gated_delta(x, 0, G * D, n_qk, x[:, n_qk + H * V:], 0, H, A.to(device), bias.to(device), H, G, D, V, st["s"],
                                  seq_ops.get_step(), q_scale=0.37).reshape(x.shape[0], H * V)
    outs = run_cut(None, hs, CUTS, device, dtype, D, caches, forward=step)
    for o, r in zip(outs, refs):
        near(o, r, dtype, f32=5e-5, bf16=5e-5)      # (the operands hold their values exactly: the recurrence is float32)


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("H,G,N,V", OUTER_SIZES)
def test_state_space_operator(device, dtype, H, G, N, V):
    g = gen(H * 11 + N)
    A, bias = forget(g, H)
    skip = rnd(g, H)
    hs = [torch.cat([rnd(g, n, H * V + 2 * G * N, dtype=dtype), rnd(g, n, H, s=4.0, dtype=dtype)], 1) for n in LENGTHS]
    refs, of = [], torch.arange(H) // (H // G)
    for h in hs:
        n = h.shape[0]
        x, B, C, dt = h.to(F64).split([H * V, G * N, G * N, H], 1)
        refs.append(O.state_space(x.reshape(n, H, V), B.reshape(n, G, N)[:, of], C.reshape(n, G, N)[:, of], O.softplus(dt + bias.to(F64)),
                                  A.to(F64), skip.to(F64))[0].reshape(n, H * V))
    st = {}

    def caches(blocks, slots):
        st["s"] = torch.empty(slots, H, N, V, device=device)
        stale(st["s"], g)

    def step(x):
        return hy_ops.state_space(x, 0, H * V, H * V + G * N, x, H * V + 2 * G * N, A.to(device), bias.to(device), skip.to(device), H, G, N, V,
                                  st["s"], seq_ops.get_step()).reshape(x.shape[0], H * V)
    outs = run_cut(None, hs, CUTS, device, dtype, N, caches, forward=step)
    for o, r in zip(outs, refs):
        near(o, r, dtype, f32=5e-5, bf16=5e-5)


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("sizes", [[1], [2], [7, 1], [17], [260]])
def test_states_that_hardly_forget_through_portions(device, dtype, sizes):
    """The first tokens' keys are asked for by the last tokens: a state that is lost, doubled or decayed twice between
    portions shows, and so does a read-out before the token's own write (the last query is the last key)."""
    g = gen(3)
    H, G, D, V, n = 2, 1, 24, 20, 260
    q, k, v = rnd(g, n, D, dtype=dtype), rnd(g, n, D, s=0.05, dtype=dtype), rnd(g, n, H * V, dtype=dtype)
    k[:3] = torch.eye(D)[:3].to(dtype) * 2
    q[-4:] = torch.eye(D)[[0, 1, 2, 3]].to(dtype)
    k[-1] = torch.eye(D)[3].to(dtype)
    k[3:-1, :4] = 0                            # nothing between overwrites what lies under the first keys
    pre = torch.cat([torch.full((n, H), 6.0), torch.full((n, H), -9.0)], 1).to(dtype)
    h = torch.cat([q, k, v, pre], 1)
    A, bias = torch.full((H,), -1.0), torch.zeros(H)
    ref, _ = O.gated_delta(q.to(F64)[:, None].expand(n, H, D) / torch.sqrt((q.to(F64) ** 2).sum(-1) + 1e-6)[:, None, None],
                           O.unit(k.to(F64))[:, None].expand(n, H, D), v.to(F64).view(n, H, V), torch.sigmoid(pre[:, :H].to(F64)),
                           torch.exp(-O.softplus(pre[:, H:].to(F64))))
    assert (ref[-4] - v[0].to(F64).view(H, V)).abs().max() < 0.2 and (ref[-1] - v[-1].to(F64).view(H, V)).abs().max() < 0.2
    st = {}

    def caches(blocks, slots):
        st["s"] = torch.empty(slots, H, D, V, device=device)
        stale(st["s"], g)
    cuts, left = [], n
    while left:
        cuts.append(min(left, sizes[len(cuts) % len(sizes)]))
        left -= cuts[-1]
    out, = run_cut(None, [h], [cuts], device, dtype, 0, caches, forward=lambda x: hy_ops.gated_delta(
        x, 0, D, 2 * D, x, 2 * D + H * V, 2 * D + H * V + H, A.to(device), bias.to(device), H, G, D, V, st["s"],
        seq_ops.get_step()).reshape(x.shape[0], H * V))
    near(out, ref.reshape(n, H * V), dtype, f32=5e-5, bf16=5e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["delta", "space"])
@pytest.mark.parametrize("H,G,D,V,copies", [(2, 1, 64, 32, 1), (3, 3, 128, 32, 1), (4, 2, 128, 128, 1), (6, 2, 64, 160, 1), (4, 2, 128, 128, 3),
                                            (4, 4, 64, 64, 5)])
def test_portions_by_chunks_equal_the_walk(monkeypatch, kind, H, G, D, V, copies):
    """32 tokens at a time and token after token: portions around one and two chunks, new ones and ones that continue a state, rows that
    are a column slice (and one too little aligned for chunks).  Both are float32 sums of exact operands: from the float64 recurrence
    they are within 16 roundings of 2^-24 in norm (D / 64 terms per lane and fold, up to four chunks' states).  A token that is
    not finite leaves the tokens in front of it and the other portions as they are.  Copies of the portions: workgroups of 64 value channels."""
    g = gen(D + V + H)
    lens, of = [1, 31, 32, 33, 64, 2, 65, 97] * copies, torch.arange(H) // (H // G)
    starts = [0, 40, 0, 7, 0, 3, 9, 0] * copies
    assert (len(lens) * H * (V // 32) > 256) == (copies > 1)
    n, n_qk = sum(lens), 2 * G * D
    wide = rnd(g, n, n_qk + H * V + 16, dtype=torch.bfloat16)
    pre = rnd(g, n, 2 * H, s=2.0, dtype=torch.bfloat16).cuda()
    A, bias = forget(g, H)
    skip = rnd(g, H)
    ctx, _ = batch(list(zip(starts, lens)), device="cuda", seed=3)
    state0 = rnd(g, max(int(s) for s in ctx.seq_slot) + 2, H, D, V)
    cuda = [t.cuda() for t in (A, bias, skip)]

    def run(rows, least):
        monkeypatch.setattr(hy_ops, "CHUNKS_MIN_TOKENS", {D: least} if least else {})
        st = state0.cuda()
        if kind == "delta":
            o = hy_ops.gated_delta(rows, 0, G * D, n_qk, pre, 0, H, *cuda[:2], H, G, D, V, st, ctx, q_scale=0.37)
        else:
            o = hy_ops.state_space(rows, n_qk, 0, G * D, pre, 0, *cuda, H, G, D, V, st, ctx)
        return o, st
    rows = wide.cuda()[:, 8:8 + n_qk + H * V]
    walk, chunks = run(rows, 0), run(rows, 1)
    off = torch.zeros(n, wide.shape[1] + 3, dtype=torch.bfloat16, device="cuda")
    off[:, 3:] = wide
    off = off[:, 11:11 + n_qk + H * V]
    odd = run(off, 1)
    assert [hy_ops._outer_chunked(r, (0, G * D, n_qk), D, V, ctx) for r in (rows, off)] == [True, False]
    x, p, at = wide[:, 8:].to(F64), pre.cpu().to(F64), 0
    for b, (start, length) in enumerate(zip(starts, lens)):
        h, pb, slot = x[at:at + length], p[at:at + length], int(ctx.seq_slot[b])
        a, c = (h[:, i * G * D:(i + 1) * G * D].reshape(length, G, D) for i in (0, 1))
        v = h[:, n_qk:n_qk + H * V].reshape(length, H, V)
        s0 = state0[slot].to(F64) if start else torch.zeros(H, D, V, dtype=F64)
        if kind == "delta":
            ref, s_ref = O.gated_delta((O.unit(a) * 0.37)[:, of], O.unit(c)[:, of], v, torch.sigmoid(pb[:, :H]),
                                       torch.exp(A.to(F64) * O.softplus(pb[:, H:] + bias.to(F64))), s0)
        else:
            ref, s_ref = O.state_space(v, a[:, of], c[:, of], O.softplus(pb[:, :H] + bias.to(F64)), A.to(F64), skip.to(F64), s0)
        for o, st in (walk, chunks, odd):
            assert (o[at:at + length].cpu().to(F64) - ref).norm() <= 16 * 2 ** -24 * ref.norm()
            assert (st[slot].cpu().to(F64) - s_ref).norm() <= 16 * 2 ** -24 * s_ref.norm()
        at += length
    at = n - 97 + 50                                                    # one token of the last portion's second chunk
    for column, value in ((n_qk + 5, float("inf")), (3, float("nan")), (G * D + 1, float("inf"))):
        bad = rows.clone()
        bad[at, column] = value
        o = run(bad, 1)[0]
        assert torch.equal(o[:at], chunks[0][:at]) and not torch.isfinite(o[at, 0]).all()
        if column > n_qk:                                               # a value channel: the others don't notice
            keep = torch.ones(H * V, dtype=torch.bool)
            keep[5] = False
            assert torch.equal(o.view(n, -1)[:, keep], chunks[0].view(n, -1)[:, keep]) and not torch.isfinite(o[at:, 0, 5]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["delta", "space"])
@pytest.mark.parametrize("H,D,V", [(24, 64, 64), (12, 128, 96)])
def test_long_portions_by_chunks_keep_every_chunks_results(monkeypatch, kind, H, D, V):
    """Portions of 8 to 47 chunks on more workgroups than the chip runs at once, several times: a wave hands its partner a chunk's strengths and the
    state's part of its results, and those of another chunk in their place are an error of the size of the results.  Every chunk's rows are within 32 roundings of 2^-24 of the walk's in norm (either is within 16 of the exact sums), and
    every run gives the same bits."""
    g = gen(H + D)
    lens = [1500, 256, 1023, 777, 1337, 288, 640, 1024] * 3
    n = sum(lens)
    rows = rnd(g, n, 2 * D + H * V, dtype=torch.bfloat16).cuda()
    pre = rnd(g, n, 2 * H, s=2.0, dtype=torch.bfloat16).cuda()
    A, bias = (t.cuda() for t in forget(g, H))
    skip = rnd(g, H).cuda()
    ctx, _ = batch([(0, m) for m in lens], device="cuda", seed=1)
    slots = max(int(s) for s in ctx.seq_slot) + 1

    def run(least):
        monkeypatch.setattr(hy_ops, "CHUNKS_MIN_TOKENS", {D: least} if least else {})
        st = torch.zeros(slots, H, D, V, device="cuda")
        if kind == "delta":
            return hy_ops.gated_delta(rows, 0, D, 2 * D, pre, 0, H, A, bias, H, 1, D, V, st, ctx, q_scale=0.37)
        return hy_ops.state_space(rows, 2 * D, 0, D, pre, 0, A, bias, skip, H, 1, D, V, st, ctx)
    walk, first = run(0).double(), run(1)
    at = 0
    for m in lens:
        for t in range(at, at + m, 32):
            e = min(t + 32, at + m)
            assert (first[t:e].double() - walk[t:e]).norm() <= 32 * 2 ** -24 * walk[t:e].norm()
        at += m
    for _ in range(10):
        assert torch.equal(run(1), first)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["delta", "space"])
@pytest.mark.parametrize("D,V", [(64, 64), (128, 64), (128, 128)])
def test_chunk_walks_of_two_and_four_waves_agree(kind, D, V):
    """Workgroups have 32 value channels up to 256 of them and 64 beyond: a column's sums are the same, so the bits are.  Portions of one,
    two, three and four chunks, the last ones whole and of a single token (each takes another turn of the buffers)."""
    g = gen(D + V)
    H, lens = 4, [128, 65, 96, 64, 97, 33, 128, 32]
    n = sum(lens)
    rows, pre = rnd(g, n, 2 * D + H * V, dtype=torch.bfloat16).cuda(), rnd(g, n, 2 * H, s=2.0, dtype=torch.bfloat16).cuda()
    A, bias, skip = (t.cuda() for t in (*forget(g, H), rnd(g, H)))
    outs = []
    few = 256 // (H * (V // 32) * len(lens))                            # copies of the batch that 256 workgroups of two hold
    for copies in (1, few, few + 1):
        ctx, _ = batch([(0, m) for m in lens] * copies, device="cuda", seed=2)
        st = torch.full((max(int(s) for s in ctx.seq_slot) + 1, H, D, V), 7.0, device="cuda")
        x, p = rows.repeat(copies, 1), pre.repeat(copies, 1)
        assert hy_ops._outer_chunked(x, (0, D, 2 * D), D, V, ctx)
        if kind == "delta":
            o = hy_ops.gated_delta(x, 0, D, 2 * D, p, 0, H, A, bias, H, 1, D, V, st, ctx)
        else:
            o = hy_ops.state_space(x, 2 * D, 0, D, p, 0, A, bias, skip, H, 1, D, V, st, ctx)
        outs.append((o.view(copies, n, H, V), st[ctx.seq_slot.long()].view(copies, len(lens), H, D, V)))
    for o, st in outs:
        assert torch.isfinite(o).all() and (o == outs[0][0]).all() and (st == outs[0][1]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,V", [(32, 64), (64, 128), (128, 64), (256, 72)])
def test_recurrence_forms_agree(dtype, D, V):
    """Small and large batches take different numbers of columns per thread, unaligned rows other fetches, single tokens another
    kernel; each gives the same result."""
    g = gen(D + V)
    H, G, n = 4, 2, 21
    rows, pre = rnd(g, n, 2 * G * D + H * V, dtype=dtype).cuda(), rnd(g, n, 2 * H, dtype=dtype).cuda()
    A, bias, skip = (t.cuda() for t in (*forget(g, H), rnd(g, H)))
    for kind in ("delta", "space"):
        def run(r, p, st, ctx):
            if kind == "delta":
                return hy_ops.gated_delta(r, 0, G * D, 2 * G * D, p, 0, H, A, bias, H, G, D, V, st, ctx)
            return hy_ops.state_space(r, 2 * G * D, 0, G * D, p, 0, A, bias, skip, H, G, D, V, st, ctx)
        outs = []
        for B in (1, 300):
            ctx, _ = batch([(0, n)] * B, device="cuda", seed=B)
            st = torch.full((B + 2, H, D, V), 7.0, device="cuda")
            o = run(rows.repeat(B, 1), pre.repeat(B, 1), st, ctx).view(B, n, H, V)
            assert torch.equal(o[0], o[-1]) and torch.equal(st[int(ctx.seq_slot[0])], st[int(ctx.seq_slot[-1])])
            outs.append((o[0], st[int(ctx.seq_slot[0])]))
        wide = torch.zeros(n, rows.shape[1] + 3, dtype=dtype, device="cuda")
        wide[:, 3:] = rows
        st = torch.full((3, H, D, V), 7.0, device="cuda")
        ctx, _ = batch([(0, n)], device="cuda")
        o = run(wide[:, 3:], pre, st, ctx)
        outs.append((o, st[int(ctx.seq_slot[0])]))
        st, steps = torch.full((3, H, D, V), 7.0, device="cuda"), []
        for t in range(n):
            ctx, _ = batch([(t, 1)], device="cuda", slots=[1])
            steps.append(run(rows[t:t + 1], pre[t:t + 1], st, ctx))
        outs.append((torch.cat(steps), st[1]))
        for o, s in outs[1:]:
            near(o, outs[0][0].cpu().to(F64), torch.float32, f32=1e-5)
            near(s, outs[0][1].cpu().to(F64), torch.float32, f32=1e-5)


# ------------------------------------------------------------------------------------------ gated norms
@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("H,D", [(1, 1), (3, 20), (5, 33), (2, 256), (1, 2052), (4, 640), (70, 8), (1, 5000)])
def test_gated_norm_forms(device, dtype, H, D):
    """sigmoid or SiLU, in front of the norm or behind it, a weight per channel or shared by the heads, a factor, results into a
    column slice."""
    g = gen(H + D)
    T, eps = 5, 1e-3
    o, wide = rnd(g, T, H, D), rnd(g, T, H * D + 5, s=2.0, dtype=dtype)
    gate = wide.to(device)[:, 5:]
    for shared in (False, True):
        w = 1 + rnd(g, D if shared else H * D, s=0.3, dtype=dtype)
        for act in (hy_ops.GATE_SIGMOID, hy_ops.GATE_SILU):
            for first in (False, True):
                a = wide[:, 5:].to(F64).view(T, H, D)
                a = O.silu(a) if act else torch.sigmoid(a)
                z = o.to(F64)
                r = O.rms(z * a, eps) if first else O.rms(z, eps) * a
                r = (r * w.to(F64).view(-1, D) * 0.7).reshape(T, H * D)
                into = torch.zeros(T, H * D + 4, dtype=dtype, device=device)
                got = hy_ops.delta_gate_norm(o.to(device), gate, w.to(device), eps, dtype, act, first, into[:, 4:], 0.7)
                near(got, r, dtype)
                assert got.data_ptr() == into[:, 4:].data_ptr() and not into[:, :4].any()


# ------------------------------------------------------------------------------------------ soft-capped windowed attention
ATT_SIZES = [(1, 1, 8, 8, 5), (4, 2, 16, 24, 64), (6, 3, 33, 7, 40), (8, 2, 64, 128, 65), (4, 4, 128, 64, 1), (2, 1, 136, 72, 63), (3, 1, 24, 40, 300)]


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("H,G,D,V,window", ATT_SIZES)
def test_soft_capped_windows_and_output_gate(device, dtype, H, G, D, V, window):
    """Scores of which many lie beyond the cap; results gated, scaled and left in a column slice; both kernel forms."""
    g = gen(H + D + window)
    cap, scale = 3.0, 2.0 * D ** -0.5
    hs = [rnd(g, n, H * D + G * D + G * V + H * V, dtype=dtype) for n in LENGTHS]
    nq = H * D + G * D + G * V
    refs = []
    for h in hs:
        n, x = h.shape[0], h.to(F64)
        r = O.window_attention(x[:, :H * D].reshape(n, H, D), x[:, H * D:H * D + G * D].reshape(n, G, D),
                               x[:, H * D + G * D:nq].reshape(n, G, V), scale, cap, window).reshape(n, H * V)
        refs.append(r * torch.sigmoid(x[:, nq:]) * 0.6)
    for force in ((False, True) if device == "cuda" and dtype == torch.bfloat16 else (False,)):
        st = {}

        def caches(blocks, slots):
            st["k"] = torch.empty(blocks, 64, G, D, dtype=dtype, device=device)
            st["v"] = torch.empty(blocks, 64, G, V, dtype=dtype, device=device)
            stale(st["k"], g)
            stale(st["v"], g)

        def step(x):
            ctx = seq_ops.get_step()
            q = hy_ops.qkv_prepare(x[:, :nq], H, G, D, V, None, None, 1e-5, None, False, ctx, st["k"], st["v"])
            into = torch.zeros(x.shape[0], H * V + 8, dtype=dtype, device=device)
            return hy_ops.paged_attention(q, st["k"], st["v"], ctx, scale, window=window, softcap=cap, gate=x[:, nq:], out=into[:, 8:],
                                          out_scale=0.6, force_rows=force)
        outs = run_cut(None, hs, CUTS, device, dtype, D, caches, forward=step)
        for o, r in zip(outs, refs):
            near(o, r, dtype)


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("window", [3, 64, 100])
@pytest.mark.parametrize("cap", [8.0, 60.0])
def test_window_edges_show(device, dtype, window, cap):
    """One key stands out for every query, exactly as far back as the window reaches, and one just outside of it stands out
    more: a window that is a token off changes the row.  Prompt rows in every form and decoded tokens; the edge passes
    page and tile borders; the largest scores reach the cap."""
    g = gen(window)
    H, G, D, V, n = 2, 1, 128, 64, 210
    q, k, v = rnd(g, n, H, D, s=0.05), rnd(g, n, G, D, s=0.05), rnd(g, n, G, V, dtype=dtype)
    # channel c of a key marks its position mod 127; a query looks for the marks of the two positions at its edge
    for j in range(n):
        k[j, :, j % 127] += 1
        if j - (window - 1) >= 0:
            q[j, :, (j - (window - 1)) % 127] += 40
        if j - window >= 0:
            q[j, :, (j - window) % 127] += 55
    q, k = q.to(dtype), k.to(dtype)
    ref = O.window_attention(q.to(F64), k.to(F64), v.to(F64), 0.4, cap, window)
    for off in (window - 1, window + 1):
        assert (O.window_attention(q.to(F64), k.to(F64), v.to(F64), 0.4, cap, off) - ref)[window + 1:].abs().amax((1, 2)).min() > 0.3
    h = torch.cat([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1)], 1)
    for cuts in ([n], [150] + [1] * 60, [61, 2, 3, 1, 80, 63]):
        for force in ((False, True) if device == "cuda" and dtype == torch.bfloat16 else (False,)):
            st = {}

            def caches(blocks, slots):
                st["k"] = torch.empty(blocks, 64, G, D, dtype=dtype, device=device)
                st["v"] = torch.empty(blocks, 64, G, V, dtype=dtype, device=device)
                stale(st["k"], g)
                stale(st["v"], g)

            def step(x):
                ctx = seq_ops.get_step()
                qq = hy_ops.qkv_prepare(x, H, G, D, V, None, None, 1e-5, None, False, ctx, st["k"], st["v"])
                return hy_ops.paged_attention(qq, st["k"], st["v"], ctx, 0.4, window=window, softcap=cap, force_rows=force)
            out, = run_cut(None, [h], [cuts], device, dtype, window, caches, forward=step)
            near(out, ref.reshape(n, H * V), dtype)


@pytest.mark.parametrize("device,dtype", CASES)
def test_soft_cap_beside_sinks_chunks_and_pooled_blocks(device, dtype):
    """The cap with what other designs ask of the same kernels: a sink (not capped), kept first tokens, a chunked mask, pooled
    blocks, and no window at all; gates behind each."""
    g = gen(5)
    H, G, D, V, n, cap, pool = 4, 2, 32, 32, 150, 2.0, 16
    h = rnd(g, n, H * D + G * D + G * V, s=1.5, dtype=dtype)
    gate, sink = rnd(g, n, H * V, dtype=dtype), rnd(g, H)
    x = h.to(F64)
    q, k, v = x[:, :H * D].reshape(n, H, D), x[:, H * D:H * D + G * D].reshape(n, G, D), x[:, H * D + G * D:].reshape(n, G, V)
    i = torch.arange(n)
    low = i[:, None] >= i[None, :]
    masks = {"plain": low, "kept": low & ((i[:, None] - i[None, :] < 40) | (i[None, :] < 3)), "chunk": low & (i[:, None] // 48 == i[None, :] // 48),
             "pooled": low & (i[:, None] - i[None, :] < 40)}
    for name, ok in masks.items():
        ref = torch.zeros(n, H, V, dtype=F64)
        for hh in range(H):
            s = cap * torch.tanh((q[:, hh] @ k[:, hh // 2].T) * 0.3 / cap).masked_fill(~ok, float("-inf"))
            s = s.masked_fill(~ok, float("-inf"))
            vals = v[:, hh // 2]
            if name == "pooled":
                e = n // pool
                kp, vp = (t[:e * pool, hh // 2].reshape(e, pool, -1).mean(1) for t in (k, v))
                if dtype == torch.bfloat16:
                    kp, vp = kp.to(dtype).to(F64), vp.to(dtype).to(F64)
                sp = cap * torch.tanh((q[:, hh] @ kp.T) * 0.3 / cap)
                last = torch.arange(e) * pool + pool - 1
                s = torch.cat([s, sp.masked_fill(last[None, :] > i[:, None] - 40, float("-inf"))], 1)
                vals = torch.cat([vals, vp])
            else:
                s = torch.cat([s, sink[hh].to(F64).expand(n, 1)], 1)
                vals = torch.cat([vals, torch.zeros(1, V, dtype=F64)])
            ref[:, hh] = torch.softmax(s, -1) @ vals
        ref = ref.reshape(n, H * V) * torch.sigmoid(gate.to(F64))
        both = torch.cat([h, gate], 1)
        for cuts in ([n], [100] + [1] * 50):
            st = {}

            def caches(blocks, slots):
                rows = hy_ops.pool_rows_per_page(64, pool)
                for key, shape in (("k", (blocks, 64, G, D)), ("v", (blocks, 64, G, V)), ("kp", (blocks, rows, G, D)), ("vp", (blocks, rows, G, V))):
                    st[key] = torch.empty(shape, dtype=dtype, device=device)
                    stale(st[key], g)

            def step(t):
                ctx = seq_ops.get_step()
                qq = hy_ops.qkv_prepare(t[:, :h.shape[1]], H, G, D, V, None, None, 1e-5, None, False, ctx, st["k"], st["v"])
                kw = {}
                if name == "pooled":
                    hy_ops.pool_blocks(st["k"], st["v"], st["kp"], st["vp"], pool, ctx)
                    kw = dict(window=40, pooled=(st["kp"], st["vp"], pool))
                else:
                    kw = dict(sink=sink.to(device), window=40 if name == "kept" else 0, keep_first=3 if name == "kept" else 0,
                              chunk=48 if name == "chunk" else 0)
                return hy_ops.paged_attention(qq, st["k"], st["v"], ctx, 0.3, softcap=cap, gate=t[:, h.shape[1]:], **kw)
            out, = run_cut(None, [both], [cuts], device, dtype, 1, caches, forward=step)
            near(out, ref, dtype)


# ------------------------------------------------------------------------------------------ layers
def delta_layer(width, m, dtype, device, g):
    """(module, its tensors under the checkpoint's names)."""
    H, G, D, V, K = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"]
    p = {}
    for n, c in (("q", G * D), ("k", G * D), ("v", H * V)):
        p[f"mix.{n}"], p[f"mix.{n}.conv"] = rnd(g, c, width, s=width ** -0.5, dtype=dtype), rnd(g, c, K, s=0.6, dtype=dtype)
    p.update({"mix.b": rnd(g, H, width, s=width ** -0.5, dtype=dtype), "mix.a": rnd(g, H, width, s=width ** -0.5, dtype=dtype),
              "mix.A_log": rnd(g, H, dtype=dtype), "mix.dt_bias": (rnd(g, H) - 1).to(dtype), "mix.norm": 1 + rnd(g, V, s=0.3, dtype=dtype),
              "mix.g": rnd(g, H * V, width, s=width ** -0.5, dtype=dtype), "mix.o": rnd(g, width, H * V, s=(H * V) ** -0.5, dtype=dtype)})
    mod = module(dtype, lambda: GatedDelta(width, H, G, D, V, K, 1e-4))
    for n in ("q", "k", "v", "g", "b", "a"):
        mod.in_proj.data[slice(*mod.rows[n])] = p[f"mix.{n}"]
    for n in "qkv":
        mod.conv.weight.data[slice(*mod.rows[n])] = p[f"mix.{n}.conv"]
    mod.A.data = -torch.exp(p["mix.A_log"].float())
    mod.dt_bias.data, mod.out_norm.data, mod.o_proj.data = p["mix.dt_bias"].float(), p["mix.norm"], p["mix.o"]
    return mod.to(device), p


def attention_layer(width, m, dtype, g):
    H, G, D, V, K = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"]
    p = {}
    for n, c in (("q", H * D), ("k", G * D), ("v", G * V)):
        p[f"mix.left.{n}"], p[f"mix.left.{n}.b"] = rnd(g, c, width, s=width ** -0.5, dtype=dtype), rnd(g, c, s=0.5, dtype=dtype)
        p[f"mix.left.{n}.conv"] = rnd(g, c, K, s=0.6, dtype=dtype)
    p.update({"mix.left.g": rnd(g, H * V, width, s=width ** -0.5, dtype=dtype), "mix.left.o": rnd(g, width, H * V, s=(H * V) ** -0.5, dtype=dtype)})
    mod = module(dtype, lambda: PagedRotaryAttention(width, H, G, D, V, m["scale"], 1e-4, m["rot"]["dims"], m["rot"]["base"],
                                                     window=m["mask"]["size"], softcap=m["softcap"], bias=True, taps=K, out_gate=True))
    return mod, p


def fill_attention(mod, p):
    g = mod.gate_rows
    mod.qkv_proj.data[:g] = p["mix.left.g"]
    mod.qkv_proj.data[g:] = torch.cat([p[f"mix.left.{n}"] for n in "qkv"])
    mod.proj_bias.data[g:] = torch.cat([p[f"mix.left.{n}.b"] for n in "qkv"])
    mod.conv.weight.data.copy_(torch.cat([p[f"mix.left.{n}.conv"] for n in "qkv"]))
    mod.o_proj.data.copy_(p["mix.left.o"])


def space_layer(width, m, dtype, g):
    H, V, N, G, K = m["heads"], m["vdim"], m["state"], m["groups"], m["conv"]
    inner, cc = H * V, H * V + 2 * G * N
    p = {"in": rnd(g, inner + cc + H, width, s=width ** -0.5, dtype=dtype), "conv": rnd(g, cc, K, s=0.6, dtype=dtype),
         "conv.b": rnd(g, cc, s=0.5, dtype=dtype), "dt_bias": (rnd(g, H) - 1).to(dtype), "A_log": rnd(g, H, dtype=dtype),
         "D": 1 + rnd(g, H, s=0.3, dtype=dtype), "norm": 1 + rnd(g, inner, s=0.3, dtype=dtype), "o": rnd(g, width, inner, s=inner ** -0.5, dtype=dtype)}
    mod = module(dtype, lambda: StateSpaceDual(width, H, V, N, G, K, m["norm_groups"], 1e-4))
    return mod, {"mix.right." + k: v for k, v in p.items()}


def fill_space(mod, p):
    p = {k[10:]: v for k, v in p.items() if k.startswith("mix.right.")}
    mod.place_in_proj(p["in"])
    mod.A.data = -torch.exp(p["A_log"].float())
    mod.dt_bias.data, mod.D.data = p["dt_bias"].float(), p["D"].float()
    for dst, k in ((mod.conv.weight, "conv"), (mod.conv.bias, "conv.b"), (mod.out_norm, "norm"), (mod.o_proj, "o")):
        dst.data.copy_(p[k])


def f64(p):
    return {k: v.to(F64) for k, v in p.items()}


DELTAS = [dict(heads=1, kv_heads=1, dim=4, vdim=4, conv=1), dict(heads=6, kv_heads=2, dim=16, vdim=24, conv=4),
          dict(heads=4, kv_heads=4, dim=24, vdim=8, conv=2), dict(heads=3, kv_heads=1, dim=33, vdim=9, conv=5)]
LEFTS = [dict(heads=1, kv_heads=1, dim=8, vdim=8, conv=1, scale=0.3, softcap=5.0, rot=dict(dims=8, base=100.0), mask=dict(size=1)),
         dict(heads=4, kv_heads=2, dim=16, vdim=40, conv=4, scale=0.5, softcap=2.0, rot=dict(dims=8, base=1000.0), mask=dict(size=33)),
         dict(heads=6, kv_heads=2, dim=24, vdim=16, conv=3, scale=0.4, softcap=20.0, rot=dict(dims=24, base=10000.0), mask=dict(size=200)),
         dict(heads=3, kv_heads=3, dim=7, vdim=5, conv=2, scale=0.6, softcap=1.0, rot=dict(dims=2, base=50.0), mask=dict(size=64))]
RIGHTS = [dict(heads=1, vdim=4, state=1, groups=1, conv=4, norm_groups=1), dict(heads=4, vdim=16, state=24, groups=2, conv=4, norm_groups=4),
          dict(heads=6, vdim=8, state=16, groups=1, conv=1, norm_groups=3), dict(heads=4, vdim=9, state=11, groups=4, conv=5, norm_groups=2)]


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("m", DELTAS, ids=lambda m: "h%d_%dx%d_taps%d" % (m["heads"], m["dim"], m["vdim"], m["conv"]))
def test_gated_delta_layer(monkeypatch, device, dtype, m):
    g = gen(m["heads"] + m["dim"])
    mod, p = delta_layer(48, m, dtype, device, g)
    hs = [rnd(g, n, 48, dtype=dtype) for n in LENGTHS]
    refs = [O.delta_mixer(h.to(F64), f64(p), m, 1e-4) for h in hs]

    def caches(blocks, slots):
        mod.allocate_state(slots, dtype, device)
        stale(mod.state, g)
        stale(mod.conv.state, g)
    for split in (1 << 30, 3):                 # one first product, and the per-head rows in a product of their own
        monkeypatch.setattr(gated_delta, "SPLIT_TOKENS", split)
        for o, r in zip(run_cut(mod, hs, CUTS, device, dtype, 1, caches), refs):
            near(o, r, dtype, f32=1e-4, bf16=4e-2)


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("k", range(4))
def test_attention_and_state_space_layers_alone(device, dtype, k):
    g = gen(30 + k)
    att, pa = attention_layer(40, LEFTS[k], dtype, g)
    fill_attention(att, pa)
    spc, ps = space_layer(40, RIGHTS[k], dtype, g)
    fill_space(spc, ps)
    hs = [rnd(g, n, 40, dtype=dtype) for n in LENGTHS]
    for mod, ref in ((att.to(device), lambda h: O.attention_mixer(h, f64(pa), LEFTS[k])),
                     (spc.to(device), lambda h: O.state_space_mixer(h, f64(ps), RIGHTS[k], 1e-4))):
        def caches(blocks, slots):
            mod.allocate_state(slots, dtype, device)
            stale(mod.conv.state, g)
            if mod is att:
                mod.allocate(blocks, 64, dtype, device)
                stale(mod.k_cache, g)
                stale(mod.v_cache, g)
            else:
                stale(mod.state, g)
        for h, o in zip(hs, run_cut(mod, hs, CUTS, device, dtype, 2, caches)):
            near(o, ref(h.to(F64)), dtype, f32=1e-4, bf16=4e-2)


@pytest.mark.parametrize("device,dtype", CASES)
@pytest.mark.parametrize("k,j", [(0, 0), (1, 1), (2, 1), (3, 3), (1, 2), (0, 3), (2, 0)])
def test_mixer_pair(device, dtype, k, j):
    """Equal and unequal taps (the joined convolution pads the shorter ones), sizes whose product needs padding rows; factors
    of both sides (bfloat16: norms over as few as four channels bring rounding of a small result up with it); and the pair the other way round, whose convolutions stay apart."""
    g = gen(50 + 4 * k + j)
    width = 40
    att, pa = attention_layer(width, LEFTS[k], dtype, g)
    spc, ps = space_layer(width, RIGHTS[j], dtype, g)
    pair = MixerPair(att, spc, 0.6, 1.7)
    assert pair.joined
    fill_attention(att, pa)                    # (after the merge: parameters are views into the merged storage)
    fill_space(spc, ps)
    m = dict(left=LEFTS[k], right=RIGHTS[j], left_scale=0.6, right_scale=1.7)
    hs = [rnd(g, n, width, dtype=dtype) for n in LENGTHS]
    refs = [O.parallel_mixer(h.to(F64), f64({**pa, **ps}), m, 1e-4) for h in hs]

    def run(mod):
        def caches(blocks, slots):
            mod.allocate_state(slots, dtype, device)
            att.allocate(blocks, 64, dtype, device)
            stale(att.k_cache, g)
            stale(att.v_cache, g)
            stale(spc.state, g)
            for c in ([mod.conv] if mod.joined else [att.conv, spc.conv]):
                stale(c.state, g)
        return run_cut(mod, hs, CUTS, device, dtype, 3, caches)

    def to_device(mod):
        """The merged tensors are no parameters of the pair: everything moves together (the engine builds on the device)."""
        for t in ("w_first", "w_last", "bias"):
            if getattr(mod, t) is not None:
                setattr(mod, t, getattr(mod, t).to(device))
        return mod.to(device)
    for o, r in zip(run(to_device(pair)), refs):
        near(o, r, dtype, f32=1e-4, bf16=8e-2)
    assert pair.state_bytes_per_slot(2) == spc.heads * spc.vdim * spc.states * 4 + \
        2 * max(pair.conv.taps - 1, 1) * (att.conv.weight.shape[0] + spc.conv.weight.shape[0])
    att, _ = attention_layer(width, LEFTS[k], dtype, g)
    spc, _ = space_layer(width, RIGHTS[j], dtype, g)
    other = MixerPair(spc, att, 1.7, 0.6)
    assert not other.joined
    fill_attention(att, pa)
    fill_space(spc, ps)
    for o, r in zip(run(to_device(other)), refs):
        near(o, r, dtype, f32=1e-4, bf16=8e-2)
