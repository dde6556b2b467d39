"""Operators of libhymix behind torch tensors: what sits between the matrix products of a decoder that mixes rotary
attention layers (sinks, sliding windows with kept first tokens, value mixing between layers) with delta-rule recurrent
layers, on a float32 residual whose sublayers are normalised on both sides, gated, and read a token-shifted input.
One kernel launch each on the current stream; the step's batch is a nanovllm.seq_ops.StepContext.  CPU tensors go to
plain-torch counterparts (nanovllm/cpu_ops.py): engine plumbing on a host without a GPU, never a fallback for a GPU tensor."""
import torch

from nanovllm import _hymix as HM
from nanovllm import cpu_ops
from nanovllm.seq_ops import StepContext


def _dev(t):
    return HM.stream_ptr(t.device)


def _rows(t, name):
    """A matrix whose rows may be a column slice of a wider product: unit stride inside a row."""
    if t.dim() != 2 or t.stride(1) != 1:
        raise HM.QLinearError(f"{name} must be a matrix with contiguous rows")
    return t


def embed_scaled(ids, embed, scale):
    """x f32 [T, W] = embed[id] * scale."""
    if not embed.is_cuda:
        return cpu_ops.embed_scaled(ids, embed, scale)
    T, W = ids.numel(), embed.shape[1]
    x = torch.empty((T, W), dtype=torch.float32, device=embed.device)
    HM.check(HM.load().hm_embed_scaled(HM.dtype_code(embed.dtype), ids.data_ptr(), embed.data_ptr(), float(scale), x.data_ptr(),
                                       T, W, _dev(embed)))
    return x


def sublayer_close(x, y, gate, gate_bias, post_w, mult, next_w, eps, dtype, carry=None):
    """The boundary between two sublayers on a float32 residual x [T, W], per token in one launch:
      y given:      x <- x + mult * rms_norm(y * sigmoid(gate + gate_bias)) * post_w      (gate: pre-activation, rows may
                    be a column slice of a wider product)
      next_w given: returns rms_norm(x) * next_w in ``dtype`` (the next sublayer's input)
      carry = (src [T, W], state [slots, layers, W], layer, ctx): state[slot of the sequence, layer] <- src[last token of
                    the sequence's portion] (what a token shift of that layer reads at the next step)."""
    if not x.is_cuda:
        return cpu_ops.sublayer_close(x, y, gate, gate_bias, post_w, mult, next_w, eps, dtype, carry)
    T, W = x.shape
    h = torch.empty((T, W), dtype=dtype, device=x.device) if next_w is not None else None
    if y is not None:
        HM.require_cuda(y, dtype, "y")
        _rows(gate, "gate")
    src = state = None
    tok_seq = qstart = seq_slot = None
    slot_stride = 0
    if carry is not None:
        src, st, layer, ctx = carry
        HM.require_cuda(src, dtype, "carry source")
        assert st.dtype == dtype and st.is_contiguous() and st.shape[2] == W
        state, slot_stride = st[:, layer], st.stride(0)
        tok_seq, qstart, seq_slot = ctx.tok_seq, ctx.qstart, ctx.seq_slot
    HM.check(HM.load().hm_sublayer_close(HM.dtype_code(dtype), x.data_ptr(), HM.ptr(y), HM.ptr(gate),
                                         gate.stride(0) if gate is not None else 0, HM.ptr(gate_bias), HM.ptr(post_w), float(mult),
                                         HM.ptr(next_w), float(eps), HM.ptr(h), HM.ptr(src), HM.ptr(state), slot_stride,
                                         HM.ptr(tok_seq), HM.ptr(qstart), HM.ptr(seq_slot), T, W, _dev(x)))
    return h


def token_shift(h, mu, state, layer, ctx: StepContext):
    """h [T, W] -> h + (h_prev - h) * mu, h_prev = the previous token's h: the row above inside a portion, the sequence's
    carried row state[slot, layer] at a portion's start, zero at position 0 (a slot is never cleared)."""
    if not h.is_cuda:
        return cpu_ops.token_shift(h, mu, state, layer, ctx)
    HM.require_cuda(h, mu.dtype, "h")
    T, W = h.shape
    out = torch.empty_like(h)
    st = state[:, layer]
    HM.check(HM.load().hm_token_shift(HM.dtype_code(h.dtype), h.data_ptr(), mu.data_ptr(), st.data_ptr(), state.stride(0),
                                      ctx.tok_seq.data_ptr(), ctx.tok_pos.data_ptr(), ctx.qstart.data_ptr(),
                                      ctx.seq_slot.data_ptr(), out.data_ptr(), T, W, _dev(h)))
    return out


def rotary_inv_freq(dims, base, device):
    """f_i = base^(-2i/dims), i < dims/2, evaluated in float64 and kept in float32."""
    i = torch.arange(dims // 2, dtype=torch.float64)
    return (float(base) ** (-2.0 * i / dims)).to(torch.float32).to(device)


def rotary_table(dims, base, device, scaling=None):
    """(frequencies f32 [dims/2], factor on every cosine and sine).  Without ``scaling``: f_i = base^(-2i/dims) and 1.
    ``scaling`` = {factor, original, fast, slow} stretches the table for contexts longer than ``original`` positions: a
    pair that makes fewer than ``slow`` turns over ``original`` positions has its frequency divided by ``factor``, one that
    makes more than ``fast`` turns keeps it, and between them a linear ramp over the pair index blends the two (the ramp
    runs from pair lo = floor(d(fast)) to hi = ceil(d(slow)), d(t) = dims ln(original / (2 pi t)) / (2 ln base), clamped
    to the table); cosines and sines grow by 0.1 ln(factor) + 1.  Evaluated in float64, kept in float32."""
    import math
    i = torch.arange(dims // 2, dtype=torch.float64)
    f = float(base) ** (-2.0 * i / dims)
    mag = 1.0
    if scaling:
        factor, orig = float(scaling["factor"]), float(scaling["original"])

        def pair_of(turns):
            return dims * math.log(orig / (2 * math.pi * turns)) / (2 * math.log(float(base)))
        lo = max(math.floor(pair_of(float(scaling["fast"]))), 0)
        hi = min(math.ceil(pair_of(float(scaling["slow"]))), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f = f / factor * ramp + f * (1 - ramp)
        mag = 0.1 * math.log(factor) + 1.0
    return f.to(torch.float32).to(device), mag


def qkv_prepare(qkv, H, G, D, V, q_norm_w, k_norm_w, eps, inv_freq, unit_norm, ctx: StepContext, k_cache, v_cache,
                v_first=None, lam=None, q_head_w=None, k_head_w=None, q_head_scale=None, interleaved=False, rot_mag=1.0,
                v_unit_norm=False):
    """From the merged product qkv [T, H*D + G*D + G*V] of a step's tokens, in one launch per token:
      q_norm_w / k_norm_w given: RMS norm over the WHOLE q (k) projection with that weight;
      rotation of the first 2 * len(inv_freq) channels of every q and k head by position * inv_freq (channel i paired
      with channel i + len(inv_freq)), angles in float32;
      unit_norm: every rotated head of q and k divided by its RMS;
      v_first given: v <- (1 - lam) v + lam v_first (lam: float32 scalar on the device);
      k and v are stored at the tokens' cache rows; returns q [T, H, D].
    q_head_w / k_head_w [D]: before the rotation every q (k) head is divided by its own RMS and multiplied by that row,
    shared by the heads; q_head_scale f32 [H]: query head h times its number after that.  inv_freq None: no rotation.
    k_cache None: qkv holds q only [T, H*D] (the layer reads another layer's keys and values); nothing is stored.
    interleaved: channel 2i pairs with 2i + 1 instead; rot_mag multiplies every cosine and sine; v_unit_norm: every value
    head is divided by its RMS (no weight) before it is stored."""
    if not qkv.is_cuda:
        return cpu_ops.qkv_prepare(qkv, H, G, D, V, q_norm_w, k_norm_w, eps, inv_freq, unit_norm, ctx, k_cache, v_cache,
                                   v_first, lam, q_head_w, k_head_w, q_head_scale, interleaved, rot_mag, v_unit_norm)
    _rows(qkv, "qkv")
    T = qkv.shape[0]
    if k_cache is None:
        assert qkv.shape[1] == H * D and v_cache is None
    else:
        assert qkv.shape[1] == H * D + G * D + G * V and k_cache.dtype == v_cache.dtype == qkv.dtype
        assert k_cache.shape[2:] == (G, D) and v_cache.shape[2:] == (G, V)
    assert inv_freq is None or inv_freq.dtype == torch.float32
    assert q_head_scale is None or q_head_scale.dtype == torch.float32
    if v_first is not None:
        _rows(v_first, "v_first")
        assert v_first.shape == (T, G * V) and lam.dtype == torch.float32
    q = torch.empty((T, H, D), dtype=qkv.dtype, device=qkv.device)
    HM.check(HM.load().hm_qkv_prepare(HM.dtype_code(qkv.dtype), qkv.data_ptr(), qkv.stride(0), H, G, D, V, HM.ptr(q_norm_w),
                                      HM.ptr(k_norm_w), float(eps), HM.ptr(inv_freq), inv_freq.numel() if inv_freq is not None else 0,
                                      int(bool(unit_norm)), ctx.tok_pos.data_ptr(), ctx.slot_mapping.data_ptr(), HM.ptr(k_cache),
                                      HM.ptr(v_cache), HM.ptr(v_first), v_first.stride(0) if v_first is not None else 0, HM.ptr(lam),
                                      q.data_ptr(), T, HM.ptr(q_head_w), HM.ptr(k_head_w), HM.ptr(q_head_scale),
                                      int(bool(interleaved)), float(rot_mag), int(bool(v_unit_norm)), _dev(qkv)))
    return q


def pool_rows_per_page(block_size, pool):
    """Rows of a pooled cache page: block e of a sequence (the mean of its tokens e*pool .. e*pool + pool - 1) is row
    e % rows of the page block_table[e // rows]; rows * pool >= block_size, so that page is the sequence's by the time
    the block is complete."""
    return (block_size + pool - 1) // pool


def pool_blocks(k_cache, v_cache, kp_cache, vp_cache, pool, ctx: StepContext):
    """For every block of ``pool`` tokens that the step completes: the block's mean key and mean value, as the caches hold
    them, into the pooled caches [blocks, pool_rows_per_page, G, D | V].  Call it after the step's keys
    and values are stored."""
    if not k_cache.is_cuda:
        return cpu_ops.pool_blocks(k_cache, v_cache, kp_cache, vp_cache, pool, ctx)
    bs, G, D, V = k_cache.shape[1], k_cache.shape[2], k_cache.shape[3], v_cache.shape[3]
    assert kp_cache.shape[1] == vp_cache.shape[1] == pool_rows_per_page(bs, pool) and kp_cache.dtype == k_cache.dtype
    HM.check(HM.load().hm_pool_blocks(HM.dtype_code(k_cache.dtype), k_cache.data_ptr(), v_cache.data_ptr(), kp_cache.data_ptr(),
                                      vp_cache.data_ptr(), ctx.block_tables.data_ptr(), ctx.seq_pos0.data_ptr(),
                                      ctx.ctx_lens.data_ptr(), ctx.num_seqs, int(ctx.max_q), G, D, V, bs, ctx.block_tables.shape[1],
                                      int(pool), kp_cache.shape[1], _dev(k_cache)))


USE_TILES = True       # bf16 attention on the matrix cores where the shape allows (tests compare both forms)


def paged_attention(q, k_cache, v_cache, ctx: StepContext, scale, sink=None, window=0, keep_first=0, force_rows=False,
                    pooled=None, chunk=0, sigmoid=False, head_bias=None, softcap=0.0, gate=None, out=None, out_scale=1.0):
    """q [T, H, D] over the paged caches k [blocks, block_size, G, D], v [blocks, block_size, G, V]; query head h reads
    key/value head h // (H/G).  The token at position i sees key j <= i, and with window > 0 only if i - j < window or
    j < keep_first.  ``sink`` f32 [H]: one more term exp(sink[h]) in the softmax denominator, without a value (zeros
    = a sink of score 0).  Scores and weights are float32.  Returns [T, H * V].
    ``pooled`` = (kp_cache, vp_cache, pool) with window > 0: beside its window the token also sees one key and value for
    every block of ``pool`` tokens whose last token lies at or before i - window (the block means pool_blocks keeps), in the
    same softmax.
    ``chunk`` > 0: the token at position i sees key j <= i only if i // chunk == j // chunk (chunks of positions counted from
    the sequence's start).  ``sigmoid``: the weight of a visible key is sigmoid(score + head_bias[h]) (f32 [H], None = 0),
    not normalised over the keys.  ``softcap`` > 0 (softmax weights): a score s becomes softcap * tanh(s / softcap).
    The result is multiplied by ``out_scale`` and, element by element, by sigmoid(``gate``) ([T, H * V], rows may be a column
    slice); ``out`` [T, H * V] (may be a column slice) takes it."""
    if not q.is_cuda:
        r = cpu_ops.paged_attention(q, k_cache, v_cache, ctx, scale, sink, window, keep_first, pooled, chunk, sigmoid, head_bias,
                                    softcap, gate, out_scale)
        return r if out is None else out.copy_(r)
    kp, vp, pool = pooled if pooled is not None else (None, None, 0)
    pr = kp.shape[1] if kp is not None else 0
    assert head_bias is None or head_bias.dtype == torch.float32
    HM.require_cuda(q, k_cache.dtype, "q")
    T, H, D = q.shape
    bs, G, V = k_cache.shape[1], k_cache.shape[2], v_cache.shape[3]
    mb = ctx.block_tables.shape[1]
    o = torch.empty((T, H * V), dtype=q.dtype, device=q.device) if out is None else _rows(out, "out")
    assert o.shape == (T, H * V) and o.dtype == q.dtype
    if gate is not None:
        _rows(gate, "gate")
        assert gate.shape == (T, H * V) and gate.dtype == q.dtype
    gs = gate.stride(0) if gate is not None else H * V
    ptail = (HM.ptr(kp), HM.ptr(vp), int(pool), int(pr), int(chunk), HM.ptr(head_bias), int(bool(sigmoid)), float(softcap or 0.0),
             o.stride(0), HM.ptr(gate), gs, float(out_scale))
    lib = HM.load()
    tiles_ok = (USE_TILES and not force_rows and q.dtype == torch.bfloat16 and D % 8 == 0 and V % 8 == 0 and D <= 128 and
                V <= 128 and bs % 64 == 0 and o.stride(0) % 4 == 0 and gs % 4 == 0 and
                (o.data_ptr() | (gate.data_ptr() if gate is not None else 0)) % 8 == 0)
    if tiles_ok and ctx.max_q == 1 and H // G <= 32:
        keys = min(mb * bs, window + keep_first + 128) if window > 0 else mb * bs
        if chunk > 0:
            keys = min(keys, chunk + 64)
        if pool:
            keys = min(mb * bs, keys + mb * bs // pool + 64)
        splits = decode_splits(ctx.num_seqs * G, keys)
        ws, n = HM.decode_workspace.get(q.device, lib.hm_attn_decode_workspace_bytes(T, H, V, splits))
        HM.check(lib.hm_attn_decode(q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), ctx.block_tables.data_ptr(),
                                    ctx.ctx_lens.data_ptr(), HM.ptr(sink), int(window), int(keep_first), float(scale), o.data_ptr(),
                                    T, H, G, D, V, bs, mb, splits, ws, n, *ptail, _dev(q)))
        return o
    if tiles_ok:
        HM.check(lib.hm_attn_tiles(q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), ctx.block_tables.data_ptr(),
                                   ctx.qstart.data_ptr(), ctx.seq_pos0.data_ptr(), HM.ptr(sink), int(window), int(keep_first),
                                   float(scale), o.data_ptr(), ctx.num_seqs, ctx.max_q, H, G, D, V, bs, mb, *ptail, _dev(q)))
        return o
    HM.check(lib.hm_attn_rows(HM.dtype_code(q.dtype), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                              ctx.block_tables.data_ptr(), ctx.tok_seq.data_ptr(), ctx.tok_pos.data_ptr(), HM.ptr(sink),
                              int(window), int(keep_first), float(scale), o.data_ptr(), T, H, G, D, V, bs, mb, *ptail, _dev(q)))
    return o


def group_norm_residual(x, y, post_w, groups, eps, dtype, next_w=None, ids=None, want_h=True, w_add=0.0, pos=None, pos_table=None):
    """The boundary between two sublayers of a float32 residual x [T, W] that is normalised on the sublayers' OUTPUT (and,
    with next_w, on their input too), the RMS norm taken over ``groups`` equal consecutive parts of the vector; per token in
    one launch, with w' = w + w_add (w_add = 1: weights stored around zero):
      y given:        x <- x + group_norm(y) * post_w'   (ids given: x <- group_norm(y[ids]) * post_w', y an embedding table,
                      without post_w y[ids] itself; x may then be None and is made here)
      pos_table:      with ids, pos_table[pos] is added (pos int32 [T])
      want_h:         returns group_norm(x) * next_w' if next_w is given, else x itself, in ``dtype`` (what the next
                      sublayer, or the vocabulary product, reads); for float32 without next_w that is x, no copy.
    Returns (x, h)."""
    on_cpu = not (y if y is not None else x).is_cuda
    if on_cpu:
        return cpu_ops.group_norm_residual(x, y, post_w, groups, eps, dtype, next_w, ids, want_h, w_add, pos, pos_table)
    T = ids.numel() if ids is not None else (y if y is not None else x).shape[0]
    W = (y if y is not None else x).shape[1]
    if x is None:
        x = torch.empty((T, W), dtype=torch.float32, device=y.device)
    if y is not None:
        HM.require_cuda(y, dtype, "y")
    if pos_table is not None:
        HM.require_cuda(pos_table, dtype, "pos_table")
        assert pos.dtype == torch.int32 and pos.numel() == T and pos_table.shape[1] == W
    h = None
    if want_h and (next_w is not None or dtype != torch.float32):
        h = torch.empty((T, W), dtype=dtype, device=x.device)
    HM.check(HM.load().hm_group_norm_residual(HM.dtype_code(dtype), x.data_ptr(), HM.ptr(y), HM.ptr(ids), HM.ptr(pos),
                                              HM.ptr(pos_table), HM.ptr(post_w), HM.ptr(next_w), float(w_add), int(groups), float(eps),
                                              HM.ptr(h), T, W, _dev(x)))
    return x, (h if h is not None or not want_h else x)


def scale_softcap_(logits, scale, cap):
    """logits f32, in place: cap * tanh(logits * scale / cap) (cap <= 0 or None: logits * scale)."""
    if not logits.is_cuda:
        return cpu_ops.scale_softcap_(logits, scale, cap)
    assert logits.dtype == torch.float32 and logits.is_contiguous()
    HM.check(HM.load().hm_scale_softcap(logits.data_ptr(), logits.numel(), float(scale), float(cap or 0.0), _dev(logits)))
    return logits


def decode_splits(num_groups, max_keys):
    """Splits of the key tiles in decode attention: about four workgroups per CU, at least two 64-key tiles per split.
    Depends only on the batch size and the cache geometry, never on the sequences' lengths."""
    want = max(1, 1024 // max(1, num_groups))
    return int(max(1, min(want, (max_keys + 127) // 128, 64)))


def delta_prepare(proj, cols, w2, w0, a_bias, H, D, decay_scale, unit_eps=1e-6):
    """The float32 inputs of a delta-rule recurrence from the mixer's merged product.  cols = ((offset, size) of r, k, the
    removal gate's pre-activation, and the decay's inner activation z) in proj's columns.  Per token, head and channel:
      decay = exp(-decay_scale * sigmoid(w2 tanh(z) + w0)),  a = sigmoid(a_pre + a_bias),  u = k / sqrt(sum k^2 + unit_eps)
    Returns f32 [T, H, 5, D] = decay, a * u, u, k, r."""
    if not proj.is_cuda:
        return cpu_ops.delta_prepare(proj, cols, w2, w0, a_bias, H, D, decay_scale)
    _rows(proj, "proj")
    T = proj.shape[0]
    (r_off, _), (k_off, _), (a_off, _), (z_off, rank) = cols
    assert w2.shape == (H * D, rank) and w2.is_contiguous() and w2.dtype == proj.dtype
    prep = torch.empty((T, H, 5, D), dtype=torch.float32, device=proj.device)
    HM.check(HM.load().hm_delta_prepare(HM.dtype_code(proj.dtype), proj.data_ptr(), proj.stride(0), r_off, k_off, a_off, z_off,
                                        w2.data_ptr(), w0.data_ptr(), a_bias.data_ptr(), rank, float(decay_scale), float(unit_eps),
                                        prep.data_ptr(), T, H, D, _dev(proj)))
    return prep


def delta_recurrence(prep, v, state, ctx: StepContext):
    """Generalized delta rule over every sequence's portion, token after token, per head with a float32 state S [D, D]:
      S <- diag(decay) S - (a u)(u^T S) + k v^T  (both terms read the old S),  o = S^T r.
    state f32 [slots, H, D, D] is read at a portion's start (zero at position 0) and left at its end.  v [T, H*D] may be a
    column slice.  Returns o f32 [T, H, D]."""
    if not prep.is_cuda:
        return cpu_ops.delta_recurrence(prep, v, state, ctx)
    _rows(v, "v")
    T, H, _, D = prep.shape
    assert state.dtype == torch.float32 and state.is_contiguous() and state.shape[1:] == (H, D, D)
    o = torch.empty((T, H, D), dtype=torch.float32, device=prep.device)
    HM.check(HM.load().hm_delta_recurrence(HM.dtype_code(v.dtype), prep.data_ptr(), v.data_ptr(), v.stride(0), state.data_ptr(),
                                           ctx.qstart.data_ptr(), ctx.seq_pos0.data_ptr(), ctx.seq_slot.data_ptr(), o.data_ptr(),
                                           ctx.num_seqs, H, D, max(int(ctx.max_q), 1), _dev(prep)))
    return o


GATE_SIGMOID, GATE_SILU = 0, 1


def delta_gate_norm(o, g, norm_w, eps, dtype, act=GATE_SIGMOID, gate_first=False, out=None, scale=1.0):
    """o f32 [T, H, D] -> every head divided by its RMS, times norm_w ([H*D], or [D] shared by the heads), times act(g) (g
    [T, H*D], rows may be a column slice), times ``scale``, in ``dtype``.  ``gate_first``: o is gated before the norm instead
    of after it.  ``out`` [T, H*D] (may be a column slice) takes the result."""
    T, H, D = o.shape
    if not o.is_cuda:
        r = cpu_ops.delta_gate_norm(o, g, norm_w, eps, dtype, act, gate_first, scale)
        return r if out is None else out.copy_(r)
    _rows(g, "g")
    if out is None:
        out = torch.empty((T, H * D), dtype=dtype, device=o.device)
    _rows(out, "out")
    assert o.is_contiguous() and g.dtype == norm_w.dtype == out.dtype == dtype and out.shape == g.shape == (T, H * D)
    assert norm_w.numel() in (D, H * D)
    HM.check(HM.load().hm_delta_gate_norm(HM.dtype_code(dtype), o.data_ptr(), g.data_ptr(), g.stride(0), norm_w.data_ptr(),
                                          int(norm_w.numel() == D), int(act), int(bool(gate_first)), float(eps), float(scale),
                                          out.data_ptr(), out.stride(0), T, H, D, _dev(o)))
    return out


# Tokens of the longest portion from which a step takes 32 tokens at a time, by key channels, where the portions have half of that on
# average: below, the chunks cost more than they save (microseconds, chunks / walk, 16 heads of 128 x 128: 1 portion of 16 10.6 / 11.7,
# of 32 10.6 / 16.7, of 128 15.7 / 46.6; 64 portions of 16 43 / 59, of 32 48 / 97; 4 heads of 64 x 64: 1 portion of 16 9.5 / 8.9, of
# 32 9.5 / 12.5; 64 of 16 10.8 / 10.7, of 32 11.0 / 14.5; state space, 16 heads of 128 x 64, 1 portion of 16 8.2 / 10.6).
CHUNKS_MIN_TOKENS = {64: 32, 128: 16}


def _outer_chunked(rows, offsets, D, V, ctx):
    """Whether a step's portions take the form of 32 tokens at a time (bf16 rows whose parts start on 16 bytes, 64 or 128 key
    channels, 32 or a multiple of it value channels; long enough)."""
    least = CHUNKS_MIN_TOKENS.get(D, 0)
    return (rows.dtype == torch.bfloat16 and 0 < least <= ctx.max_q and 2 * rows.shape[0] >= least * ctx.num_seqs and V % 32 == 0 and
            rows.data_ptr() % 16 == 0 and all(c % 8 == 0 for c in (rows.stride(0), *offsets)) and ctx.num_seqs <= 65535)


def _outer_work(rows, H, ctx):
    n = HM.load().hm_outer_chunk_work_bytes(rows.shape[0], ctx.num_seqs, H)
    return torch.empty((n,), dtype=torch.uint8, device=rows.device)


def _outer_args(rows, pre, state, o_shape, H, D, V, ctx):
    """Checks of the outer-product recurrences; the output."""
    _rows(rows, "rows")
    _rows(pre, "pre")
    T = rows.shape[0]
    assert pre.shape[0] == T and pre.dtype == rows.dtype
    assert state.dtype == torch.float32 and state.is_contiguous() and state.shape[1:] == (H, D, V)
    return torch.empty(o_shape, dtype=torch.float32, device=rows.device)


def _outer_gates(rows, H, ctx):
    """Scratch for the gates of a walk that takes token after token."""
    return torch.empty((rows.shape[0], H, 8), dtype=torch.float32, device=rows.device) if ctx.max_q > 1 else None


def gated_delta(rows, q_off, k_off, v_off, pre, b_off, a_off, A, dt_bias, H, G, D, V, state, ctx: StepContext, q_scale=1.0,
                unit_eps=1e-6):
    """Gated delta rule over every sequence's portion, token after token, per head with a float32 state S [D, V]:
      S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q,
    g = exp(A softplus(a + dt_bias)), beta = sigmoid(b), k and q unit vectors (x / sqrt(sum x^2 + unit_eps)), q times q_scale.
    ``rows`` [T, *] holds q, k (G groups of D channels; head h reads group h // (H/G)) and v (H heads of V) at their columns,
    ``pre`` [T, *] b and a (one per head); both may be column slices.  A, dt_bias f32 [H].  state f32 [slots, H, D, V] is read
    at a portion's start (zero at position 0) and left at its end.  Returns o f32 [T, H, V]."""
    if not rows.is_cuda:
        return cpu_ops.gated_delta(rows, q_off, k_off, v_off, pre, b_off, a_off, A, dt_bias, H, G, D, V, unit_eps, q_scale, state, ctx)
    assert A.dtype == dt_bias.dtype == torch.float32 and A.numel() == dt_bias.numel() == H
    o = _outer_args(rows, pre, state, (rows.shape[0], H, V), H, D, V, ctx)
    if _outer_chunked(rows, (q_off, k_off, v_off), D, V, ctx):
        work = _outer_work(rows, H, ctx)
        HM.check(HM.load().hm_gated_delta_chunks(rows.data_ptr(), rows.stride(0), q_off, k_off, v_off, pre.data_ptr(), pre.stride(0), b_off,
                                                 a_off, A.data_ptr(), dt_bias.data_ptr(), float(unit_eps), float(q_scale),
                                                 None, work.data_ptr(), state.data_ptr(), ctx.qstart.data_ptr(),
                                                 ctx.seq_pos0.data_ptr(), ctx.seq_slot.data_ptr(), o.data_ptr(), ctx.num_seqs,
                                                 rows.shape[0], H, G, D, V, int(ctx.max_q), _dev(rows)))
        return o
    gates = _outer_gates(rows, H, ctx)
    HM.check(HM.load().hm_gated_delta(HM.dtype_code(rows.dtype), rows.data_ptr(), rows.stride(0), q_off, k_off, v_off, pre.data_ptr(),
                                      pre.stride(0), b_off, a_off, A.data_ptr(), dt_bias.data_ptr(), float(unit_eps), float(q_scale),
                                      HM.ptr(gates), state.data_ptr(), ctx.qstart.data_ptr(), ctx.seq_pos0.data_ptr(),
                                      ctx.seq_slot.data_ptr(), o.data_ptr(), ctx.num_seqs, rows.shape[0], H, G, D, V, int(ctx.max_q),
                                      _dev(rows)))
    return o


def state_space(rows, x_off, b_off, c_off, pre, dt_off, A, dt_bias, D, H, G, N, V, state, ctx: StepContext):
    """State-space dual recurrence over every sequence's portion, per head with a float32 state S [N, V]:
      dt = softplus(dt_pre + dt_bias);  S <- exp(A dt) S + dt B x^T;  y = S^T C + D x.
    ``rows`` [T, *] holds x (H heads of V), B and C (G groups of N; head h reads group h // (H/G)) at their columns, ``pre``
    the step sizes' pre-activations (one per head).  A, dt_bias, D f32 [H].  state f32 [slots, H, N, V] as in gated_delta.
    Returns y f32 [T, H, V]."""
    if not rows.is_cuda:
        return cpu_ops.state_space(rows, x_off, b_off, c_off, pre, dt_off, A, dt_bias, D, H, G, N, V, state, ctx)
    assert A.dtype == dt_bias.dtype == D.dtype == torch.float32 and A.numel() == dt_bias.numel() == D.numel() == H
    y = _outer_args(rows, pre, state, (rows.shape[0], H, V), H, N, V, ctx)
    if _outer_chunked(rows, (x_off, b_off, c_off), N, V, ctx):
        work = _outer_work(rows, H, ctx)
        HM.check(HM.load().hm_state_space_chunks(rows.data_ptr(), rows.stride(0), x_off, b_off, c_off, pre.data_ptr(), pre.stride(0), dt_off,
                                                 A.data_ptr(), dt_bias.data_ptr(), D.data_ptr(), None, work.data_ptr(),
                                                 state.data_ptr(), ctx.qstart.data_ptr(), ctx.seq_pos0.data_ptr(),
                                                 ctx.seq_slot.data_ptr(), y.data_ptr(), ctx.num_seqs, rows.shape[0], H, G, N, V,
                                                 int(ctx.max_q), _dev(rows)))
        return y
    gates = _outer_gates(rows, H, ctx)
    HM.check(HM.load().hm_state_space(HM.dtype_code(rows.dtype), rows.data_ptr(), rows.stride(0), x_off, b_off, c_off, pre.data_ptr(),
                                      pre.stride(0), dt_off, A.data_ptr(), dt_bias.data_ptr(), D.data_ptr(), HM.ptr(gates),
                                      state.data_ptr(), ctx.qstart.data_ptr(), ctx.seq_pos0.data_ptr(), ctx.seq_slot.data_ptr(),
                                      y.data_ptr(), ctx.num_seqs, rows.shape[0], H, G, N, V, int(ctx.max_q), _dev(rows)))
    return y


def relu_squared(z, row_scale=None, out=None):
    """max(z, 0)^2, times row_scale[t] (f32 [T]) if given; z [T, F] and ``out`` may be column slices of wider matrices."""
    T, Fw = z.shape
    if out is None:
        out = torch.empty((T, Fw), dtype=z.dtype, device=z.device)
    if not z.is_cuda:
        out.copy_(cpu_ops.relu_squared(z, row_scale))
        return out
    _rows(z, "z")
    _rows(out, "out")
    assert out.shape == (T, Fw) and out.dtype == z.dtype and (row_scale is None or row_scale.dtype == torch.float32)
    HM.check(HM.load().hm_relu_squared(HM.dtype_code(z.dtype), z.data_ptr(), z.stride(0), HM.ptr(row_scale), out.data_ptr(),
                                       out.stride(0), T, Fw, _dev(z)))
    return out


def layer_norm_residual(x, y, next_w, eps, dtype, ids=None, y2=None, routed=None):
    """The boundary between two blocks of a float32 residual x [T, W] whose blocks read a layer norm (weight, no bias) of it;
    per token in one launch:
      x <- x + y + y2     (ids given: x <- y[ids], y an embedding table; x may then be None and is made here)
      routed = (prod, pair_row, weights or None), as moe_experts(combine=False) leaves it: the token's pairs are added too
                          ((y, None, None): a sum that is already there)
      next_w given:       h = (x - mean) / sqrt(mean((x - mean)^2) + eps) * next_w in ``dtype``.
    Returns (x, h)."""
    prod = pair_row = wts = None
    if routed is not None:
        if routed[1] is None:
            assert y2 is None
            y2 = routed[0]
        else:
            prod, pair_row, wts = routed
    src = y if y is not None else x
    if not src.is_cuda:
        assert prod is None
        return cpu_ops.layer_norm_residual(x, y, next_w, eps, dtype, ids, y2)
    T = ids.numel() if ids is not None else src.shape[0]
    W = src.shape[1]
    if x is None:
        x = torch.empty((T, W), dtype=torch.float32, device=src.device)
    for a, name in ((y, "y"), (y2, "y2"), (prod, "prod")):
        if a is not None:
            HM.require_cuda(a, dtype, name)
    h = torch.empty((T, W), dtype=dtype, device=x.device) if next_w is not None else None
    HM.check(HM.load().hm_layer_norm_residual(HM.dtype_code(dtype), x.data_ptr(), HM.ptr(y), HM.ptr(ids), HM.ptr(y2), HM.ptr(prod),
                                              HM.ptr(pair_row), HM.ptr(wts), pair_row.numel() // T if prod is not None else 0,
                                              HM.ptr(next_w), float(eps), HM.ptr(h), T, W, _dev(x)))
    return x, h


def selective_scan(x, dt_pre, dt_bias, bc, b_off, c_off, A, D, z, state, ctx: StepContext, out=None):
    """Selective scan over every sequence's portion, token after token, with a float32 state S [N] per channel:
      dt = softplus(dt_pre + dt_bias);  S <- exp(dt A) S + dt x B;  out = (S . C + D x) silu(z)
    x, z [T, channels] and bc (its columns b_off, c_off are B and C) may be column slices; dt_pre f32 [T, channels]; A f32
    [channels, N], dt_bias and D f32 [channels].  state f32 [slots, channels, N] is read at a portion's start (zero at
    position 0) and left at its end.  ``out`` [T, channels] (may be a column slice) takes the result."""
    T, C = x.shape
    N = A.shape[1]
    if out is None:
        out = torch.empty((T, C), dtype=x.dtype, device=x.device)
    if not x.is_cuda:
        out.copy_(cpu_ops.selective_scan(x, dt_pre, dt_bias, bc, b_off, c_off, A, D, z, state, ctx))
        return out
    for a, name in ((x, "x"), (dt_pre, "dt_pre"), (bc, "bc"), (z, "z"), (out, "out")):
        _rows(a, name)
    assert x.dtype == bc.dtype == z.dtype == out.dtype and dt_pre.dtype == A.dtype == D.dtype == dt_bias.dtype == torch.float32
    assert dt_pre.shape == z.shape == out.shape == (T, C) and A.shape == (C, N) and A.is_contiguous()
    assert dt_bias.numel() == D.numel() == C and bc.shape[0] == T and max(b_off, c_off) + N <= bc.shape[1]
    assert state.dtype == torch.float32 and state.is_contiguous() and state.shape[1:] == (C, N)
    HM.check(HM.load().hm_selective_scan(HM.dtype_code(x.dtype), x.data_ptr(), x.stride(0), dt_pre.data_ptr(), dt_pre.stride(0),
                                         dt_bias.data_ptr(), bc.data_ptr(), bc.stride(0), b_off, c_off, A.data_ptr(), D.data_ptr(),
                                         z.data_ptr(), z.stride(0), state.data_ptr(), ctx.qstart.data_ptr(), ctx.seq_pos0.data_ptr(),
                                         ctx.seq_slot.data_ptr(), out.data_ptr(), out.stride(0), ctx.num_seqs, C, N,
                                         max(int(ctx.max_q), 1), _dev(x)))
    return out


def dyt_residual(x, y, post, nxt, dtype, ids=None, want_h=True):
    """The boundary between two sublayers of a float32 residual x [T, W] whose sublayers sit between two Dynamic-Tanh
    norms, dyt(z) = tanh(alpha z) * w + b with a norm given as (w [W], b [W], alpha f32 [1]); one elementwise launch:
      y given:   x <- x + dyt_post(y)     (ids given: x <- y[ids], y an embedding table, no norm; x may be None)
      want_h:    returns dyt_nxt(x), or x itself without ``nxt``, in ``dtype``.
    Returns (x, h)."""
    src = y if y is not None else x
    if not src.is_cuda:
        return cpu_ops.dyt_residual(x, y, post, nxt, dtype, ids, want_h)
    T = ids.numel() if ids is not None else src.shape[0]
    W = src.shape[1]
    if x is None:
        x = torch.empty((T, W), dtype=torch.float32, device=src.device)
    if y is not None:
        HM.require_cuda(y, dtype, "y")
    pw, pb, pa = post if post is not None else (None, None, None)
    nw, nb, na = nxt if nxt is not None else (None, None, None)
    for a in (pa, na):
        assert a is None or a.dtype == torch.float32
    h = None
    if want_h and (nxt is not None or dtype != torch.float32):
        h = torch.empty((T, W), dtype=dtype, device=x.device)
    HM.check(HM.load().hm_dyt_residual(HM.dtype_code(dtype), x.data_ptr(), HM.ptr(y), HM.ptr(ids), HM.ptr(pw), HM.ptr(pb), HM.ptr(pa),
                                       HM.ptr(nw), HM.ptr(nb), HM.ptr(na), HM.ptr(h), T, W, _dev(x)))
    return x, (h if h is not None or not want_h else x)


def lightning_recurrence(proj, q_off, k_off, v_off, H, D, V, decay, state, ctx: StepContext):
    """Linear attention with a constant decay per head over every sequence's portion, token after token, with a float32
    state S [D, V] per head:  S <- decay[h] S + k v^T,  o = S^T q,  where q, k [T, H*D] and v [T, H*V] are silu of the
    columns q_off, k_off, v_off of proj.  state f32 [slots, H, D, V] is read at a portion's start (zero at position 0) and
    left at its end.  decay f32 [H].  Returns o f32 [T, H, V]."""
    if not proj.is_cuda:
        return cpu_ops.lightning_recurrence(proj, q_off, k_off, v_off, H, D, V, decay, state, ctx)
    _rows(proj, "proj")
    T = proj.shape[0]
    assert state.dtype == torch.float32 and state.is_contiguous() and state.shape[1:] == (H, D, V)
    assert decay.dtype == torch.float32 and decay.numel() == H
    o = torch.empty((T, H, V), dtype=torch.float32, device=proj.device)
    HM.check(HM.load().hm_lightning_recurrence(HM.dtype_code(proj.dtype), proj.data_ptr(), proj.stride(0), q_off, k_off, v_off,
                                               decay.data_ptr(), state.data_ptr(), ctx.qstart.data_ptr(), ctx.seq_pos0.data_ptr(),
                                               ctx.seq_slot.data_ptr(), o.data_ptr(), ctx.num_seqs, H, D, V,
                                               max(int(ctx.max_q), 1), _dev(proj)))
    return o
