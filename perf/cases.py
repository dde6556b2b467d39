"""Workloads of the framework by use, one pass each through its public operators and modules, with their inputs, the work
they cannot do without, and their results in 64 bits.

What a serving step spends its time in: the quantized projections of a decoder layer (one row, a decode batch, a prompt
batch; weight-only and with quantized activations; int8 and fp8; scales per row and per group), a quantized Qwen3 over a
batch of prompts, decode attention over its paged cache, and the mixers and feed-forwards of the other families in both
directions: paged attention with its windows, sinks and soft caps, latent attention, routed experts, and the recurrences over
prompts.  Sizes are those of this repository's model configurations (Qwen3 0.6B, 4B and 8B; the families' layers of 1024 and
2048 channels) and of its benchmark (prompts and contexts of 100 to about 2000 tokens, up to 256 sequences).  Decode of a
recurrence moves a state that the pass itself changes, so it is not among them: a pass here can be called again.
float32 activations exist to check models against other implementations and are represented by the recurrences alone."""
import math
import os
import sys
from types import SimpleNamespace

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "nano-vllm-hw3_amd"))

DEV, BF16, F64 = "cuda", torch.bfloat16, torch.float64
# hidden, query heads, key/value heads, head dim, feed-forward of the Qwen3 sizes
MODELS = {"0.6b": (1024, 16, 8, 128, 3072), "4b": (2560, 32, 8, 128, 9728), "8b": (4096, 32, 8, 128, 12288)}
VOCAB = 151936
QDTYPES = {"int8": torch.int8, "fp8": torch.float8_e4m3fn}
PAGE = 64                      # tokens per page of the families' caches


# ------------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one user, one token: the four projections of a Qwen3-0.6B layer on a single row (latency and launches)
        dict(name="linears_1_int8", kind="linears", model="0.6b", rows=1, quant="per_row_weight_only", dtype="int8", group=0),
        # a decode batch of Qwen3-4B with quantized activations
        dict(name="linears_64_w8a8_fp8", kind="linears", model="4b", rows=64, quant="per_row", dtype="fp8", group=0),
        # a batch of prompts of Qwen3-4B with per-group scales, a ragged row count as prompts make it
        dict(name="linears_4099_g128", kind="linears", model="4b", rows=4099, quant="per_group", dtype="int8", group=128),
        # prompts of the headline benchmark through a quantized Qwen3-0.6B (two of its layers): embedding to last-row logits
        dict(name="qwen3_prefill", kind="qwen3", model="0.6b", layers=2, seqs=12, least=100, most=1024, quant="per_row_weight_only",
             dtype="int8", group=0),
        # decode attention of the headline benchmark in the middle of its run: 131 sequences of 300 to 1800 tokens
        dict(name="qwen3_decode_attention", kind="decode_attention", seqs=131, least=300, most=1800, heads=16, kv_heads=8),
        # prompts through a windowed, soft-capped attention layer, every fourth one continuing a cached prefix
        dict(name="attention_prefill", kind="attention", seqs=8, least=900, most=1100, cached=True, heads=16, kv_heads=8, dim=128,
             window=512, keep=0, sink=False, softcap=30.0, step="prefill"),
        # a decode batch over full attention with sinks
        dict(name="attention_decode", kind="attention", seqs=64, least=700, most=1300, cached=False, heads=16, kv_heads=8, dim=128,
             window=0, keep=0, sink=True, softcap=0.0, step="decode"),
        # prompts through latent attention: cache rows of a 192-channel latent and 64 rotated channels
        dict(name="latent_prefill", kind="latent", seqs=8, least=900, most=1100, cached=True, heads=16, rank=192, rot=64, window=0,
             sink=False, step="prefill"),
        dict(name="latent_decode", kind="latent", seqs=64, least=700, most=1300, cached=False, heads=16, rank=192, rot=64, window=0,
             sink=True, step="decode"),
        # routed experts on a batch of prompts, and on a decode batch
        dict(name="experts_prefill", kind="experts", rows=8192, width=2048, ff=1536, experts=16, top=4, act="silu_glu"),
        dict(name="experts_decode", kind="experts", rows=64, width=2048, ff=1536, experts=16, top=4, act="silu_glu"),
        # prompts through a gated-delta layer of 2048 channels
        dict(name="recurrence_prefill", kind="recurrence", op="gated_delta", seqs=8, least=900, most=1100, heads=16, dim=128, vdim=128,
             rows="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lengths_range(rng, lo, hi):
    a, b = sorted((_log(rng, lo, hi), _log(rng, lo, hi)))
    return a, b


def draw(rng):
    kind = rng.choice(["linears", "linears", "qwen3", "decode_attention", "attention", "attention", "latent", "experts", "experts",
                       "recurrence"])
    if kind == "linears":
        model = rng.choice(sorted(MODELS))
        quant = rng.choice(["per_row_weight_only", "per_row", "per_group", "per_tensor"])
        most = int(8.0e11 / (2.0 * sum(n * k for n, k in _shapes(model).values())))
        return dict(kind=kind, model=model, rows=_log(rng, 1, min(8192, most)), quant=quant, dtype=rng.choice(sorted(QDTYPES)),
                    group=rng.choice([64, 128, 256]) if quant == "per_group" else 0)
    if kind == "qwen3":
        a, b = _lengths_range(rng, 20, 1024)
        quant = rng.choice(["per_row_weight_only", "per_group", "per_tensor"])
        return dict(kind=kind, model="0.6b", layers=2, seqs=rng.randint(1, 12), least=a, most=b, quant=quant,
                    dtype=rng.choice(sorted(QDTYPES)), group=128 if quant == "per_group" else 0)
    if kind == "decode_attention":
        a, b = _lengths_range(rng, 50, 1800)
        heads, kv = rng.choice([(16, 8), (32, 8)])
        return dict(kind=kind, seqs=_log(rng, 1, 128), least=a, most=b, heads=heads, kv_heads=kv)
    if kind == "attention":
        step = rng.choice(["prefill", "decode"])
        a, b = _lengths_range(rng, 100, 1100 if step == "prefill" else 1800)
        heads, kv = rng.choice([(8, 4), (16, 8), (16, 4)])
        window = rng.choice([0, 0, 256, 512])
        return dict(kind=kind, seqs=rng.randint(1, 8) if step == "prefill" else _log(rng, 1, 64), least=a, most=b,
                    cached=rng.random() < 0.5 and step == "prefill", heads=heads, kv_heads=kv, dim=rng.choice([64, 128, 128]),
                    window=window, keep=rng.choice([0, 4]) if window else 0, sink=rng.random() < 0.5,
                    softcap=rng.choice([0.0, 0.0, 30.0]), step=step)
    if kind == "latent":
        step = rng.choice(["prefill", "decode"])
        a, b = _lengths_range(rng, 100, 1100 if step == "prefill" else 1800)
        rank, rot = rng.choice([(64, 64), (128, 0), (192, 64), (256, 0)])
        return dict(kind=kind, seqs=rng.randint(1, 8) if step == "prefill" else _log(rng, 1, 64), least=a, most=b,
                    cached=rng.random() < 0.5 and step == "prefill", heads=rng.choice([8, 16]), rank=rank, rot=rot,
                    window=rng.choice([0, 0, 512]), sink=rng.random() < 0.5, step=step)
    if kind == "experts":
        width, ff = rng.choice([(1024, 768), (2048, 1536), (2048, 768)])
        return dict(kind=kind, rows=_log(rng, 1, 8000), width=width, ff=ff, experts=rng.choice([8, 16, 32]), top=rng.choice([2, 4]),
                    act=rng.choice(["silu_glu", "clamped_glu", "gelu", "relu_sq"]))
    a, b = _lengths_range(rng, 50, 1100)
    op = rng.choice(["gated_delta", "gated_delta", "state_space", "lightning", "delta", "scan"])
    heads, dim, vdim = {"gated_delta": rng.choice([(8, 128, 128), (16, 128, 128)]), "state_space": rng.choice([(16, 128, 64), (32, 128, 64)]),
                        "lightning": rng.choice([(8, 128, 128), (16, 128, 128)]), "delta": rng.choice([(16, 64, 64), (32, 64, 64)]),
                        "scan": rng.choice([(2048, 16, 1), (4096, 16, 1)])}[op]
    return dict(kind="recurrence", op=op, seqs=rng.randint(1, 8), least=a, most=b, heads=heads, dim=dim, vdim=vdim,
                rows=rng.choice(["bf16", "bf16", "f32"]))


# --------------------------------------------------------------------------------------------------------- common pieces
def _shapes(model):
    """(output, input) channels of a layer's four projections."""
    h, hq, hkv, d, ff = MODELS[model]
    return dict(qkv=((hq + 2 * hkv) * d, h), o=(h, hq * d), gate_up=(2 * ff, h), down=(h, ff))


def _lengths(case):
    """Ragged lengths between ``least`` and ``most``: part of the case, not of the seed (every seed has the same work)."""
    a, b, n = case["least"], case["most"], case["seqs"]
    return [a + (i * 7919 + 37 * i * i) % (b - a + 1) for i in range(n)]


class _Random:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)
        self.cpu = torch.Generator().manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=BF16):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def permutation(self, n):
        return torch.randperm(n, generator=self.cpu)


def _pages(lengths, page, order):
    """Pages of every sequence, drawn from the pool in the given order -> int32 [B, most pages]."""
    counts = [(n + page - 1) // page for n in lengths]
    tables = torch.zeros(len(lengths), max(counts), dtype=torch.int32)
    at = 0
    for b, c in enumerate(counts):
        tables[b, :c] = order[at:at + c].int()
        at += c
    return tables


def _portions(case):
    """(cached tokens, new tokens) of every sequence of the step."""
    lengths = _lengths(case)
    if case["step"] == "decode":
        return [(n - 1, 1) for n in lengths]
    return [(n // 2, n - n // 2) if case["cached"] and i % 4 == 3 else (0, n) for i, n in enumerate(lengths)]


def _context(portions, tables, page):
    from nanovllm.seq_ops import StepContext
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    tok_seq, tok_pos, slots, starts = [], [], [], [0]
    for b, (p, n) in enumerate(portions):
        tok_seq += [b] * n
        tok_pos += range(p, p + n)
        row = tables[b].tolist()
        slots += [row[i // page] * page + i % page for i in range(p, p + n)]
        starts.append(starts[-1] + n)
    return StepContext(tok_seq=i32(tok_seq), tok_pos=i32(tok_pos), qstart=i32(starts), seq_pos0=i32([p for p, _ in portions]),
                       ctx_lens=i32([p + n for p, n in portions]), seq_slot=i32(list(range(len(portions)))), slot_mapping=i32(slots),
                       block_tables=tables.to(DEV), num_seqs=len(portions), num_tokens=starts[-1], max_q=max(n for _, n in portions),
                       block_size=page, qstart_host=starts)


def _seen(portions, window, keep=0):
    """Query-key pairs that a causal mask with a window and kept first tokens leaves, and the cached tokens that are read."""
    pairs = keys = 0
    for p, n in portions:
        for i in range(p, p + n):
            first = max(0, i + 1 - window) if window else 0
            pairs += i + 1 - first + min(keep, first)
        first = max(0, p + 1 - window) if window else 0
        keys += p + n - first + min(keep, first)
    return pairs, keys


# ---- quantization in plain torch: what the modules hold, widened to 64 bits
def _round_away(y):
    return torch.trunc(y + torch.copysign(torch.full_like(y, 0.5), y))


def _to_fp8(y):
    """The nearest e4m3 value (ties to even, at most 448): 3 fraction bits, exponents from -6 on."""
    y = y.to(F64)
    step = torch.exp2(torch.floor(torch.log2(y.abs().clamp(min=2.0 ** -6))) - 3)
    return (torch.round(y / step) * step).clamp(-448.0, 448.0)


def _narrow(y, dtype):
    return _round_away(y).clamp(-128, 127).to(F64) if dtype == "int8" else _to_fp8(y)


def _row_quantized(x, dtype):
    amax = x.float().abs().amax(1, keepdim=True).clamp(min=1e-8)
    top = torch.full_like(amax, 127.0 if dtype == "int8" else 448.0)        # (a tensor: by a number torch multiplies with 1 / number)
    return _narrow(x.float() * (top / amax), dtype), (amax / top).to(F64)


def _dequantized(w, quant, dtype, group):
    if quant in ("per_row", "per_row_weight_only"):
        q, s = _row_quantized(w, dtype)
        return q * s
    top = torch.tensor(127.0 if dtype == "int8" else 448.0, device=DEV)
    if quant == "per_group":
        x = w.float().view(w.shape[0], -1, group)
        s = x.abs().amax(-1, keepdim=True).clamp(min=1e-8) / top
        y = x / s
    else:                                      # one scale, kept in bf16; the quotient is rounded to bf16 in front of the cast
        x = w
        s = w.abs().amax().clamp(min=1e-8) / top.to(BF16)
        y = (x / s).float()
    q = torch.round(y).clamp(-128, 127).to(F64) if dtype == "int8" else _to_fp8(y)
    return (q * s.to(F64)).view(w.shape)


def _attend(q, k, v, scale, p0, window=0, keep=0, sink=None, softcap=0.0):
    """q [t, H, D] at positions p0.., k [n, G, D], v [n, G, V] in 64 bits -> [t, H, V]."""
    t, h, _ = q.shape
    n, g, _ = k.shape
    k, v = (x.repeat_interleave(h // g, 1).transpose(0, 1).contiguous() for x in (k, v))
    s = torch.matmul(q.transpose(0, 1), k.transpose(1, 2)) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    i, j = torch.arange(p0, p0 + t, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
    seen = j <= i
    if window:
        seen &= (i - j < window) | (j < keep)
    s = s.masked_fill(~seen, float("-inf"))
    if sink is not None:
        s = torch.cat([s, sink.to(F64)[:, None, None].expand(h, t, 1)], -1)
    return torch.matmul(torch.softmax(s, -1)[..., :n], v).transpose(0, 1)


# -------------------------------------------------------------------------------------------- the quantized linear layers
def _linears_inputs(case, seed):
    r = _Random(seed)
    shapes = _shapes(case["model"])
    ws = {n: r.normal(*s, std=s[1] ** -0.5) for n, s in shapes.items()}
    xs = {n: r.normal(case["rows"], s[1]) for n, s in shapes.items()}
    return ws, xs


def _linears_prepare(case, seed):
    from nanovllm.utils import quantization as NQ
    ws, xs = _linears_inputs(case, seed)
    dt = QDTYPES[case["dtype"]]
    mods = {}
    for n, w in ws.items():
        if case["quant"] == "per_group":
            m = NQ.QGroupLinear(dt, w, None, case["group"])
        elif case["quant"] == "per_tensor":
            m = NQ.QTensorLinear(dt, w, None)
        else:
            m = NQ.QLinear(dt, w, None, weight_only=case["quant"] == "per_row_weight_only")
        if n == "gate_up":
            m.enable_silu_mul()
        mods[n] = m.tile()
    return mods, xs


def _linears_run(state):
    mods, xs = state
    return {n: m(xs[n]) for n, m in mods.items()}


def _linears_exact(case, seed):
    ws, xs = _linears_inputs(case, seed)
    out = {}
    for n, w in ws.items():
        x = xs[n].to(F64)
        if case["quant"] == "per_row":
            qx, sx = _row_quantized(xs[n], case["dtype"])
            x = qx * sx
        y = x @ _dequantized(w, case["quant"], case["dtype"], case["group"]).t()
        if n == "gate_up":
            g, u = y.chunk(2, -1)
            y = F.silu(g) * u
        out[n] = y
    return out


def _linears_work(case):
    m, nbytes, flops = case["rows"], 0, 0
    for n, (out, k) in _shapes(case["model"]).items():
        scales = out * (k // case["group"]) if case["quant"] == "per_group" else 1 if case["quant"] == "per_tensor" else out
        nbytes += out * k + 4 * scales + 2 * m * k + 2 * m * (out // 2 if n == "gate_up" else out)
        flops += 2 * m * out * k
    return dict(bytes=nbytes, flops=flops)


# ------------------------------------------------------------------------------------------- a quantized Qwen3 over prompts
def _qwen3_inputs(case, seed):
    r = _Random(seed)
    h = MODELS[case["model"]][0]
    layers = [dict({n: r.normal(*s, std=s[1] ** -0.5) for n, s in _shapes(case["model"]).items()},
                   norms=[(1.0 + 0.1 * r.normal(n, dtype=torch.float32)).to(BF16) for n in (h, h, 128, 128)])
              for _ in range(case["layers"])]
    embed = r.normal(VOCAB, h, std=0.7)
    norm = (1.0 + 0.1 * r.normal(h, dtype=torch.float32)).to(BF16)
    lengths = _lengths(case)
    ids = torch.randint(0, 10000, (sum(lengths),), generator=r.g, device=DEV)
    pages = sum((n + 255) // 256 for n in lengths) + 4
    return layers, embed, norm, lengths, ids, _pages(lengths, 256, r.permutation(pages)), pages


def _qwen3_prepare(case, seed):
    from nanovllm.models.qwen3 import AttnContext, Qwen3ForCausalLM
    from nanovllm.utils.quantization import apply_quant_from_config
    layers, embed, norm, lengths, ids, tables, pages = _qwen3_inputs(case, seed)
    h, hq, hkv, d, ff = MODELS[case["model"]]
    cfg = SimpleNamespace(hidden_size=h, num_hidden_layers=case["layers"], num_attention_heads=hq, num_key_value_heads=hkv, head_dim=d,
                          intermediate_size=ff, vocab_size=VOCAB, rms_norm_eps=1e-6, rope_theta=1000000.0, max_position_embeddings=40960,
                          tie_word_embeddings=True, attention_bias=False, hidden_act="silu")
    before = torch.get_default_dtype()
    torch.set_default_dtype(BF16)
    torch.set_default_device(DEV)
    try:
        model = Qwen3ForCausalLM(cfg)
    finally:
        torch.set_default_device("cpu")
        torch.set_default_dtype(before)
    model.model.embed_tokens.weight.data.copy_(embed)
    model.model.norm.weight.data.copy_(norm)
    for m, w in zip(model.model.layers, layers):
        for mod, n in ((m.self_attn.qkv_proj, "qkv"), (m.self_attn.o_proj, "o"), (m.mlp.gate_up_proj, "gate_up"), (m.mlp.down_proj, "down")):
            mod.weight.data.copy_(w[n])
        for mod, x in zip((m.input_layernorm, m.post_attention_layernorm, m.self_attn.q_norm, m.self_attn.k_norm), w["norms"]):
            mod.weight.data.copy_(x)
    apply_quant_from_config(model, SimpleNamespace(quant_type=case["quant"], linear_dtype=QDTYPES[case["dtype"]], group_size=case["group"]))
    cache = torch.zeros(2, case["layers"], pages, 256, hkv, d, dtype=BF16, device=DEV)
    for i, m in enumerate(model.model.layers):
        m.self_attn.k_cache, m.self_attn.v_cache = cache[0, i], cache[1, i]
    cu, pos, slots = [0], [], []
    for b, n in enumerate(lengths):
        row = tables[b].tolist()
        cu.append(cu[-1] + n)
        pos += range(n)
        slots += [row[i // 256] * 256 + i % 256 for i in range(n)]
    ctx = AttnContext(is_prefill=True, cu_seqlens=cu, slot_mapping=torch.tensor(slots, dtype=torch.int32, device=DEV),
                      cu_seqlens_dev=torch.tensor(cu, dtype=torch.int32, device=DEV), max_seqlen=max(lengths))
    return model, ids, torch.tensor(pos, device=DEV), ctx, torch.tensor(cu[1:], device=DEV) - 1, cache


def _qwen3_run(state):
    from nanovllm.models.qwen3 import set_context
    model, ids, positions, ctx, last, cache = state
    with torch.inference_mode():
        set_context(ctx)
        hidden = model(ids, positions)
        return dict(logits=model.compute_logits(hidden[last].contiguous()), cache=cache)


def _rms(x, w):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w.to(F64)


def _qwen3_exact(case, seed):
    layers, embed, norm, lengths, ids, tables, pages = _qwen3_inputs(case, seed)
    h, hq, hkv, d, ff = MODELS[case["model"]]
    pos = torch.cat([torch.arange(n, device=DEV) for n in lengths]).to(F64)
    freq = pos[:, None] / (1000000.0 ** (torch.arange(0, d, 2, dtype=F64, device=DEV) / d))
    cos, sin = freq.cos()[:, None], freq.sin()[:, None]

    def turned(x):
        a, b = x.chunk(2, -1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
    cache = torch.zeros(2, case["layers"], pages * 256, hkv, d, dtype=F64, device=DEV)
    slots = torch.cat([tables[b].long()[torch.arange(n) // 256] * 256 + torch.arange(n) % 256 for b, n in enumerate(lengths)]).to(DEV)
    res = embed[ids].to(F64)
    for i, w in enumerate(layers):
        deq = {n: _dequantized(w[n], case["quant"], case["dtype"], case["group"]) for n in _shapes(case["model"])}
        q, k, v = (_rms(res, w["norms"][0]) @ deq["qkv"].t()).split([hq * d, hkv * d, hkv * d], -1)
        q = turned(_rms(q.reshape(-1, hq, d), w["norms"][2]))
        k = turned(_rms(k.reshape(-1, hkv, d), w["norms"][3]))
        v = v.reshape(-1, hkv, d)
        cache[0, i, slots], cache[1, i, slots] = k, v
        at, outs = 0, []
        for n in lengths:
            outs.append(_attend(q[at:at + n], k[at:at + n], v[at:at + n], d ** -0.5, 0))
            at += n
        res = res + torch.cat(outs).reshape(-1, hq * d) @ deq["o"].t()
        g, u = (_rms(res, w["norms"][1]) @ deq["gate_up"].t()).chunk(2, -1)
        res = res + (F.silu(g) * u) @ deq["down"].t()
    last = torch.tensor(lengths, device=DEV).cumsum(0) - 1
    return dict(logits=_rms(res[last], norm) @ embed.to(F64).t(), cache=cache.view(2, case["layers"], pages, 256, hkv, d))


def _qwen3_work(case):
    h, hq, hkv, d, ff = MODELS[case["model"]]
    lengths = _lengths(case)
    t = sum(lengths)
    params = sum(n * k for n, k in _shapes(case["model"]).values())
    pairs = _seen([(0, n) for n in lengths], 0)[0]
    flops = case["layers"] * (2 * t * params + 4 * pairs * hq * d) + 2 * len(lengths) * VOCAB * h
    return dict(bytes=case["layers"] * (params + 4 * t * hkv * d) + 2 * VOCAB * h + 2 * t * h, flops=flops)


# ------------------------------------------------------------------------------------ decode attention of the Qwen3 models
def _decode_inputs(case, seed):
    r = _Random(seed)
    lengths = _lengths(case)
    pages = sum((n + 255) // 256 for n in lengths) + 4
    kc, vc = (r.normal(pages, 256, case["kv_heads"], 128) for _ in range(2))
    return r.normal(case["seqs"], case["heads"], 128), kc, vc, _pages(lengths, 256, r.permutation(pages)), lengths


def _decode_prepare(case, seed):
    q, kc, vc, tables, lengths = _decode_inputs(case, seed)
    return q, kc, vc, tables.to(DEV), torch.tensor(lengths, dtype=torch.int32, device=DEV)


def _decode_run(state):
    from nanovllm import ops
    return ops.paged_attn_decode(*state, 128 ** -0.5)


def _decode_exact(case, seed):
    q, kc, vc, tables, lengths = _decode_inputs(case, seed)
    out = []
    for b, n in enumerate(lengths):
        rows = tables[b, :(n + 255) // 256].long().to(DEV)
        k, v = (c[rows].reshape(-1, case["kv_heads"], 128)[:n].to(F64) for c in (kc, vc))
        out.append(_attend(q[b:b + 1].to(F64), k, v, 128 ** -0.5, n - 1))
    return torch.cat(out)


def _decode_work(case):
    keys = sum(_lengths(case))
    return dict(bytes=4 * keys * case["kv_heads"] * 128 + 4 * case["seqs"] * case["heads"] * 128, flops=4 * keys * case["heads"] * 128)


# -------------------------------------------------------------------- paged attention and latent attention of the families
def _attention_inputs(case, seed):
    r = _Random(seed)
    portions = _portions(case)
    lengths = [p + n for p, n in portions]
    pages = sum((n + PAGE - 1) // PAGE for n in lengths) + 4
    tables = _pages(lengths, PAGE, r.permutation(pages))
    rows = sum(n for _, n in portions)
    sink = r.normal(case["heads"], dtype=torch.float32) if case["sink"] else None
    if case["kind"] == "latent":
        width = case["rank"] + case["rot"]
        return portions, tables, r.normal(rows, case["heads"], width), (r.normal(pages, PAGE, width),), sink
    kc, vc = (r.normal(pages, PAGE, case["kv_heads"], case["dim"]) for _ in range(2))
    return portions, tables, r.normal(rows, case["heads"], case["dim"]), (kc, vc), sink


def _attention_prepare(case, seed):
    portions, tables, q, caches, sink = _attention_inputs(case, seed)
    return case, _context(portions, tables, PAGE), q, caches, sink


def _attention_run(state):
    from nanovllm import hy_ops, seq_ops
    case, ctx, q, caches, sink = state
    if case["kind"] == "latent":
        return seq_ops.latent_attention(q, caches[0], ctx, q.shape[2] ** -0.5, value_cols=case["rank"], window=case["window"], sink=sink)
    return hy_ops.paged_attention(q, caches[0], caches[1], ctx, case["dim"] ** -0.5, sink, case["window"], case["keep"],
                                  softcap=case["softcap"])


def _attention_exact(case, seed):
    portions, tables, q, caches, sink = _attention_inputs(case, seed)
    latent, out, at = case["kind"] == "latent", [], 0
    for b, (p, n) in enumerate(portions):
        rows = tables[b, :(p + n + PAGE - 1) // PAGE].long().to(DEV)
        kv = [c[rows].flatten(0, 1)[:p + n].to(F64) for c in caches]
        k, v = (kv[0][:, None], kv[0][:, None, :case["rank"]]) if latent else kv
        o = _attend(q[at:at + n].to(F64), k, v, q.shape[2] ** -0.5, p, case["window"], 0 if latent else case["keep"], sink,
                    0.0 if latent else case["softcap"])
        out.append(o if latent else o.flatten(1))
        at += n
    return torch.cat(out)


def _attention_work(case):
    portions = _portions(case)
    rows = sum(n for _, n in portions)
    if case["kind"] == "latent":
        pairs, keys = _seen(portions, case["window"])
        dk, dv, row = case["rank"] + case["rot"], case["rank"], case["rank"] + case["rot"]
    else:
        pairs, keys = _seen(portions, case["window"], case["keep"])
        dk, dv, row = case["dim"], case["dim"], 2 * case["kv_heads"] * case["dim"]
    return dict(bytes=2 * keys * row + 2 * rows * case["heads"] * (dk + dv), flops=2 * pairs * case["heads"] * (dk + dv))


# ---------------------------------------------------------------------------------------------------------- routed experts
GATED = ("silu_glu", "clamped_glu")


def _experts_inputs(case, seed):
    r = _Random(seed)
    e, w, f = case["experts"], case["width"], case["ff"]
    parts = 2 if case["act"] in GATED else 1
    h = r.normal(case["rows"], w)
    router, bias = r.normal(e, w, std=w ** -0.5, dtype=torch.float32), r.normal(e, std=0.5, dtype=torch.float32)
    return h, router, bias, r.normal(e, parts * f, w, std=w ** -0.5), r.normal(e, w, f, std=f ** -0.5)


def _experts_prepare(case, seed):
    from nanovllm import seq_ops
    h, router, bias, w_gu, w_down = _experts_inputs(case, seed)
    tiled = (seq_ops.tile_expert_weights(w_gu, 2 if case["act"] in GATED else 1), seq_ops.tile_expert_weights(w_down))
    return case, h, router, bias, w_gu, w_down, tiled


def _experts_run(state):
    from nanovllm import seq_ops
    case, h, router, bias, w_gu, w_down, tiled = state
    kind = dict(silu_glu=seq_ops.ACT_SILU_GLU, clamped_glu=seq_ops.ACT_CLAMPED_GLU, gelu=seq_ops.ACT_GELU,
                relu_sq=seq_ops.ACT_RELU_SQ)[case["act"]]
    limit, alpha = (7.0, 1.702) if case["act"] == "clamped_glu" else (float("inf"), 1.0)
    idx, wts = seq_ops.moe_route(h, router, case["top"], bias=bias)
    y = seq_ops.moe_experts(h, idx, wts, w_gu, w_down, limit, alpha, tiled=tiled, act_kind=kind)
    return dict(idx=idx, wts=wts, y=y)


def _experts_exact(case, seed):
    h, router, bias, w_gu, w_down = _experts_inputs(case, seed)
    x = h.to(F64)
    p = torch.softmax(x @ router.to(F64).t() + bias.to(F64), -1)
    wts, idx = p.topk(case["top"], -1)
    wts = wts / wts.sum(-1, keepdim=True)
    y = torch.zeros(h.shape, dtype=F64, device=DEV)
    for e in range(case["experts"]):
        tok, k = (idx == e).nonzero(as_tuple=True)
        z = x[tok] @ w_gu[e].to(F64).t()
        if case["act"] in GATED:
            g, u = z.chunk(2, -1)
            if case["act"] == "silu_glu":
                a = F.silu(g) * u
            else:
                g = g.clamp(max=7.0)
                a = g * torch.sigmoid(1.702 * g) * (u.clamp(-7.0, 7.0) + 1.0)
        else:
            a = F.gelu(z) if case["act"] == "gelu" else torch.relu(z).pow(2)
        y.index_add_(0, tok, wts[tok, k][:, None] * (a @ w_down[e].to(F64).t()))
    return dict(idx=None, wts=wts, y=y)


def _experts_work(case):
    t, e, w, f, top = (case[k] for k in ("rows", "experts", "width", "ff", "top"))
    mats = 3 if case["act"] in GATED else 2
    touched = e * (1.0 - (1.0 - top / e) ** t)
    return dict(bytes=int(2 * touched * mats * w * f + 4 * t * w + 4 * e * w + 8 * t * top), flops=2 * t * top * mats * w * f + 2 * t * e * w)


# --------------------------------------------------------------------------------------------- the recurrences over prompts
def _recurrence_inputs(case, seed):
    r = _Random(seed)
    lengths = _lengths(case)
    t, h, d, v = sum(lengths), case["heads"], case["dim"], case["vdim"]
    dt = BF16 if case["rows"] == "bf16" else torch.float32
    op = case["op"]
    # step sizes between 0.001 and 0.1 and rates between -1 and -16, as these layers are initialised
    step = torch.exp(r.uniform(h, lo=math.log(1e-3), hi=math.log(1e-1)))
    x = dict(dt_bias=torch.log(torch.expm1(step)), A=-r.uniform(h, lo=1.0, hi=16.0))
    if op == "gated_delta":
        x.update(rows=F.silu(r.normal(t, h * d + h * v, dtype=torch.float32)).to(dt), pre=r.normal(t, 2 * h, dtype=dt))
    elif op == "state_space":
        x.update(rows=F.silu(r.normal(t, h * v + 8 * d, dtype=torch.float32)).to(dt), pre=r.normal(t, h, dtype=dt),
                 D=r.uniform(h, lo=0.5, hi=1.5))
    elif op == "lightning":
        x.update(rows=r.normal(t, h * (2 * d + v), dtype=dt),
                 decay=torch.tensor([1.0 - 2.0 ** -(3 + 6 * i / max(1, h - 1)) for i in range(h)], device=DEV))
    elif op == "delta":
        x.update(rows=r.normal(t, 4 * h * d + 64, dtype=dt), w2=r.normal(h * d, 64, std=0.1, dtype=dt), w0=r.normal(h * d, dtype=dt),
                 a_bias=r.normal(h * d, dtype=dt))
    else:
        x.update(rows=F.silu(r.normal(t, h, dtype=torch.float32)).to(dt), z=r.normal(t, h, dtype=dt), bc=r.normal(t, 2 * d, dtype=dt),
                 dt_pre=r.normal(t, h, dtype=torch.float32), A=-torch.arange(1.0, d + 1, device=DEV).repeat(h, 1).contiguous(),
                 D=r.uniform(h, lo=0.5, hi=1.5))
    return x, lengths


def _recurrence_prepare(case, seed):
    x, lengths = _recurrence_inputs(case, seed)
    h, d, v = case["heads"], case["dim"], case["vdim"]
    ctx = _context([(0, n) for n in lengths], _pages(lengths, PAGE, torch.arange(sum((n + PAGE - 1) // PAGE for n in lengths))), PAGE)
    state = torch.zeros((len(lengths), h, d) if case["op"] == "scan" else (len(lengths), h, d, v), device=DEV)
    return case, x, ctx, state


def _recurrence_run(state):
    from nanovllm import hy_ops
    case, x, ctx, s = state
    h, d, v, op = case["heads"], case["dim"], case["vdim"], case["op"]
    rows = x["rows"]
    if op == "gated_delta":                    # a query and a key head for every two value heads
        o = hy_ops.gated_delta(rows, 0, h // 2 * d, h * d, x["pre"], 0, h, x["A"], x["dt_bias"], h, h // 2, d, v, s, ctx, q_scale=d ** -0.5)
    elif op == "state_space":
        o = hy_ops.state_space(rows, 0, h * v, h * v + 4 * d, x["pre"], 0, x["A"], x["dt_bias"], x["D"], h, 4, d, v, s, ctx)
    elif op == "lightning":
        o = hy_ops.lightning_recurrence(rows, 0, h * d, 2 * h * d, h, d, v, x["decay"], s, ctx)
    elif op == "delta":
        w = h * d
        prep = hy_ops.delta_prepare(rows, ((0, w), (w, w), (2 * w, w), (4 * w, 64)), x["w2"], x["w0"], x["a_bias"], h, d, math.exp(-0.5))
        o = hy_ops.delta_recurrence(prep, rows[:, 3 * w:4 * w], s, ctx)
    else:
        o = hy_ops.selective_scan(rows, x["dt_pre"], x["dt_bias"], x["bc"], 0, d, x["A"], x["D"], x["z"], s, ctx)
    return dict(o=o, state=s)


def _recurrence_exact(case, seed):
    x, lengths = _recurrence_inputs(case, seed)
    x = {k: a.to(F64) for k, a in x.items()}
    h, d, v, op = case["heads"], case["dim"], case["vdim"], case["op"]
    rows, t = x["rows"], x["rows"].shape[0]
    if op == "scan":
        dt = F.softplus(x["dt_pre"] + x["dt_bias"])
        item = lambda i: (torch.exp(dt[i][:, :, None] * x["A"]), (dt[i] * rows[i])[:, :, None] * x["bc"][i, None, :d], x["bc"][i, d:])  # noqa: E731
        out = torch.empty(t, h, dtype=F64, device=DEV)
    else:
        out = torch.empty(t, h, v, dtype=F64, device=DEV)
        if op == "gated_delta":
            q, k = (a.reshape(t, h // 2, d).repeat_interleave(2, 1) for a in rows[:, :h * d].chunk(2, -1))
            q, k = (a / torch.sqrt(a.pow(2).sum(-1, keepdim=True) + 1e-6) for a in (q, k))
            q, val = q * d ** -0.5, rows[:, h * d:].reshape(t, h, v)
            beta, g = torch.sigmoid(x["pre"][:, :h]), torch.exp(x["A"] * F.softplus(x["pre"][:, h:] + x["dt_bias"]))
        elif op == "state_space":
            val, k, q = rows.split([h * v, 4 * d, 4 * d], -1)
            val, (k, q) = val.reshape(t, h, v), (a.reshape(t, 4, d).repeat_interleave(h // 4, 1) for a in (k, q))
            beta = F.softplus(x["pre"] + x["dt_bias"])
            g = torch.exp(x["A"] * beta)
        elif op == "lightning":
            q, k, val = F.silu(rows).split([h * d, h * d, h * v], -1)
            q, k, val = q.reshape(t, h, d), k.reshape(t, h, d), val.reshape(t, h, v)
            beta, g = torch.ones(t, h, dtype=F64, device=DEV), x["decay"].expand(t, h)
        else:
            q, k, a, val, z = rows.split([h * d] * 4 + [64], -1)
            q, k, val = q.reshape(t, h, d), k.reshape(t, h, d), val.reshape(t, h, v)
            g = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(z) @ x["w2"].t() + x["w0"])).reshape(t, h, d)
            u = k / torch.sqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)
            beta = torch.sigmoid(a + x["a_bias"]).reshape(t, h, d) * u
    starts = torch.tensor([0] + lengths[:-1], device=DEV).cumsum(0)
    order = sorted(range(len(lengths)), key=lambda b: -lengths[b])            # longest first: the running ones are a prefix
    starts, lens = starts[torch.tensor(order, device=DEV)], [lengths[b] for b in order]
    S = torch.zeros((len(lengths), h, d) if op == "scan" else (len(lengths), h, d, v), dtype=F64, device=DEV)
    for n in range(max(lens)):
        live = sum(m > n for m in lens)
        i, s = starts[:live] + n, S[:live]
        if op == "scan":
            g_, w_, c_ = item(i)
            s.mul_(g_).add_(w_)
            out[i] = torch.einsum("bcn,bn->bc", s, c_)
            continue
        ki, vi = k[i], val[i]
        if op == "delta":
            w_ = beta[i][..., None] * torch.matmul(u[i][:, :, None, :], s)
            s.mul_(g[i][..., None]).sub_(w_).add_(ki[..., None] * vi[:, :, None, :])
        else:
            s.mul_(g[i][..., None, None])
            if op == "gated_delta":
                vi = vi - torch.matmul(ki[:, :, None, :], s)[:, :, 0]
            s.add_(ki[..., None] * (beta[i][..., None] * vi)[:, :, None, :])
        out[i] = torch.matmul(q[i][:, :, None, :], s)[:, :, 0]
    state = torch.empty_like(S)
    state[torch.tensor(order, device=DEV)] = S
    if op == "state_space":
        out = out + x["D"][:, None] * val
    if op == "scan":
        out = (out + x["D"] * rows) * F.silu(x["z"])
    return dict(o=out, state=state)


def _recurrence_work(case):
    t, b, h, d, v, op = sum(_lengths(case)), case["seqs"], case["heads"], case["dim"], case["vdim"], case["op"]
    size = 2 if case["rows"] == "bf16" else 4
    cols = dict(gated_delta=h * d + h * v + 2 * h, state_space=h * v + 8 * d + h, lightning=h * (2 * d + v), delta=4 * h * d + 64,
                scan=2 * h + 2 * d)[op]
    out = size * h if op == "scan" else 4 * h * v
    flops = dict(gated_delta=7, state_space=5, lightning=5, delta=8, scan=7)[op] * t * h * d * v
    return dict(bytes=t * (cols * size + out + (4 * h if op == "scan" else 0)) + 4 * b * h * d * v, flops=flops)


# -------------------------------------------------------------------------------------------------------- the entry points
_KINDS = {
    "linears": (_linears_prepare, _linears_run, _linears_exact, _linears_work),
    "qwen3": (_qwen3_prepare, _qwen3_run, _qwen3_exact, _qwen3_work),
    "decode_attention": (_decode_prepare, _decode_run, _decode_exact, _decode_work),
    "attention": (_attention_prepare, _attention_run, _attention_exact, _attention_work),
    "latent": (_attention_prepare, _attention_run, _attention_exact, _attention_work),
    "experts": (_experts_prepare, _experts_run, _experts_exact, _experts_work),
    "recurrence": (_recurrence_prepare, _recurrence_run, _recurrence_exact, _recurrence_work),
}


def prepare(case, seed):
    return case["kind"], _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state[0]][1](state[1])


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    """About four times what one pass is off its 64-bit result: the rounding of bf16 results (2e-3), of the bf16 values that
    the path hands on inside (attention weights, activations between two products, a layer's sublayers), or of 32-bit sums."""
    kind = case["kind"]
    if kind == "recurrence":
        return {"rel": 1e-2, "max": 0.2} if case["op"] == "scan" and case["rows"] == "bf16" else {"rel": 1e-5, "max": 1e-3}
    if kind == "qwen3":
        return {"rel": 2.5e-2, "max": 0.5}
    if kind == "experts":
        return {"rel": 1.2e-2, "max": 0.2, "differ": 1e-3}
    return {"rel": 1e-2, "max": 0.2}
