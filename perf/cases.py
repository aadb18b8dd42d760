"""Workloads of the attention hot path, as a program that uses this package issues them.

A case is a dict of plain values; `prepare` makes what the program holds before the call (KV pools, slot tables, plans,
weights), `run` is one pass through the public entry points of `parrotserve_amd.kernels`.  Lengths follow from the case
alone (its "lens" is the seed they are drawn from), contents and slot placement from the seed given to `prepare`.

Kinds
  layer   everything of a decoder layer around its library GEMMs, for a decode batch: norm, rotary + KV append, attention,
          residual add + norm, activation
  decode  shared-prefix decode over prefix groups, on the tables the attention plug-in builds once per iteration
  paged   the same through the reference-named op: one prefix, query heads that share KV heads
  ragged  decode of independent requests through the reference-named op
  prefill packed ragged chunks, each causal over a forked parent context
  ops     the element-wise passes of a decoder layer over a prefill's tokens
  move    discontinuous token move between KV pools
  sample  temperature, top-p and draw for a batch of logit rows
"""
import math
import random

import torch

from parrotserve_amd import kernels, mem

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


# --------------------------------------------------------------------------- #
# the cases
# --------------------------------------------------------------------------- #
def listed():
    return [
        # a handful of chat sessions forked from one short system prompt on a 7B model: launch latency counts
        dict(name="layer_few_sessions", kind="layer", dtype="f16", heads=32, head_dim=128, ffn=11008, batch=8, prefix=512,
             own_lo=32, own_hi=128, lens=0),
        # the headline decode step: 64 requests forked from one 4096-token prompt (7B heads)
        dict(name="decode_one_prompt", kind="decode", dtype="f16", heads=32, head_dim=128, groups=1, branches=64,
             prefix=4096, own_lo=16, own_hi=512, lens=1),
        # several applications at once: four prompts of 32 branches each, long answers (13B heads)
        dict(name="decode_four_prompts", kind="decode", dtype="f16", heads=40, head_dim=128, groups=4, branches=32,
             prefix=6000, own_lo=32, own_hi=1024, lens=4),
        # a popular application: 256 users of one 8192-token prompt, short answers so far
        dict(name="decode_many_users", kind="decode", dtype="f16", heads=32, head_dim=128, groups=1, branches=256,
             prefix=8192, own_lo=5, own_hi=64, lens=2),
        # the headline batch on a model with grouped KV heads (32 query heads over 8), bf16, reference-named op
        dict(name="paged_grouped_heads", kind="paged", dtype="bf16", heads=32, kv_heads=8, head_dim=128, branches=64,
             prefix=4096, own_lo=16, own_hi=512, lens=1),
        # nothing shared: 256 independent requests of 128 to 8192 tokens
        dict(name="ragged_256", kind="ragged", dtype="f16", heads=32, head_dim=128, batch=256, ctx_lo=128, ctx_hi=8192,
             lens=2),
        # one more turn of one conversation: a short Fill over a context of two thousand tokens
        dict(name="prefill_one_turn", kind="prefill", dtype="bf16", heads=32, head_dim=128, chunks=1, new_lo=61, new_hi=61,
             parent=1987, lens=0),
        # the headline prefill: 16 ragged chunks over forked 2048-token parents (13B heads, bf16)
        dict(name="prefill_forked_chunks", kind="prefill", dtype="bf16", heads=40, head_dim=128, chunks=16, new_lo=64,
             new_hi=1024, parent=2048, lens=3),
        # the Fill of a shared 8192-token prompt itself, no parent (13B heads)
        dict(name="prefill_shared_prompt", kind="prefill", dtype="f16", heads=40, head_dim=128, chunks=1, new_lo=8192,
             new_hi=8192, parent=0, lens=0),
        # the element-wise passes that go with the headline prefill (13B layer, bf16)
        dict(name="ops_prefill_layer", kind="ops", dtype="bf16", heads=40, head_dim=128, ffn=13824, tokens=9404, lens=3),
        # 65536 rows of 8 KB copied between random slots
        dict(name="move_64k_rows", kind="move", dtype="f16", heads=32, head_dim=128, tokens=65536, pool=131072),
        # the sampler's pass over the logits of a 64-request iteration
        dict(name="sample_64", kind="sample", dtype="f16", rows=64, vocab=32000, temperature=0.8, top_p=0.9),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["layer", "decode", "decode", "paged", "ragged", "prefill", "prefill", "ops", "move", "sample"])
    dtype = rng.choice(["f16", "bf16"])
    heads = rng.choice([32, 40])
    lens = rng.randrange(1 << 20)
    if kind == "layer":
        own_hi = _log_int(rng, 8, 512)
        return dict(kind=kind, dtype=dtype, heads=heads, head_dim=128, ffn=11008 if heads == 32 else 13824,
                    batch=_log_int(rng, 1, 64), prefix=_log_int(rng, 64, 4096), own_lo=max(1, own_hi // 16), own_hi=own_hi,
                    lens=lens)
    if kind == "decode":
        own_hi = _log_int(rng, 8, 1024)
        return dict(kind=kind, dtype=dtype, heads=heads, head_dim=128, groups=rng.choice([1, 1, 1, 2, 3, 4]),
                    branches=_log_int(rng, 2, 256), prefix=_log_int(rng, 256, 8192), own_lo=max(1, own_hi // 16),
                    own_hi=own_hi, lens=lens)
    if kind == "paged":
        own_hi = _log_int(rng, 16, 1024)
        return dict(kind=kind, dtype=dtype, heads=32, kv_heads=rng.choice([4, 8, 8, 16]), head_dim=128,
                    branches=_log_int(rng, 4, 128), prefix=_log_int(rng, 256, 8192), own_lo=max(1, own_hi // 16),
                    own_hi=own_hi, lens=lens)
    if kind == "ragged":
        return dict(kind=kind, dtype=dtype, heads=heads, head_dim=128, batch=_log_int(rng, 1, 256),
                    ctx_lo=_log_int(rng, 16, 512), ctx_hi=_log_int(rng, 512, 8192), lens=lens)
    if kind == "prefill":
        new_hi = _log_int(rng, 16, 8192)
        return dict(kind=kind, dtype=dtype, heads=heads, head_dim=128, chunks=_log_int(rng, 1, 16),
                    new_lo=max(1, new_hi // rng.choice([1, 2, 16])), new_hi=new_hi,
                    parent=rng.choice([0, _log_int(rng, 16, 6000), _log_int(rng, 16, 6000)]), lens=lens)
    if kind == "ops":
        return dict(kind=kind, dtype=dtype, heads=heads, head_dim=128, ffn=11008 if heads == 32 else 13824,
                    tokens=_log_int(rng, 16, 9404), lens=lens)
    if kind == "move":
        tokens = _log_int(rng, 256, 65536)
        return dict(kind=kind, dtype=dtype, heads=heads, head_dim=128, tokens=tokens, pool=2 * tokens)
    return dict(kind=kind, dtype=dtype, rows=_log_int(rng, 1, 128), vocab=rng.choice([32000, 50272]),
                temperature=rng.choice([0.5, 0.8, 1.0]), top_p=rng.choice([0.9, 0.95, 1.0]))


def draw(rng):
    most_bytes = max(work(c)["bytes"] for c in listed())
    most_flops = max(work(c)["flops"] for c in listed())
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= most_bytes and w["flops"] <= most_flops:
            return case


# --------------------------------------------------------------------------- #
# sizes
# --------------------------------------------------------------------------- #
def _between(case, n, lo, hi):
    r = random.Random(case["lens"])
    return [r.randint(lo, hi) for _ in range(n)]


def _contexts(case):
    r = random.Random(case["lens"])
    lo, hi = math.log(case["ctx_lo"]), math.log(case["ctx_hi"])
    return [int(round(math.exp(r.uniform(lo, hi)))) for _ in range(case["batch"])]


def _attention_work(heads, kv_heads, head_dim, rows, kv_tokens, pairs):
    """K and V rows read once, queries read and outputs written once; two products of `head_dim` per (query, key)."""
    return {"bytes": 2 * (2 * kv_tokens * kv_heads * head_dim + 2 * rows * heads * head_dim),
            "flops": 4 * heads * head_dim * pairs}


def work(case):
    kind, H = case["kind"], case.get("heads", 0)
    D = case.get("head_dim", 0)
    if kind in ("layer", "decode", "paged"):
        groups = case.get("groups", 1)
        B = case["batch"] if kind == "layer" else groups * case["branches"]
        own = sum(_between(case, B, case["own_lo"], case["own_hi"]))
        w = _attention_work(H, case.get("kv_heads", H), D, B, groups * case["prefix"] + own, B * case["prefix"] + own)
        if kind == "layer":
            w["bytes"] += _ops_bytes(B, H * D, case["ffn"])
        return w
    if kind == "ragged":
        total = sum(_contexts(case))
        return _attention_work(H, H, D, case["batch"], total, total)
    if kind == "prefill":
        new = _between(case, case["chunks"], case["new_lo"], case["new_hi"])
        P = case["parent"]
        return _attention_work(H, H, D, sum(new), len(new) * P + sum(new), sum(n * P + n * (n + 1) // 2 for n in new))
    if kind == "ops":
        return {"bytes": _ops_bytes(case["tokens"], H * D, case["ffn"]), "flops": 0}
    if kind == "move":
        return {"bytes": 2 * case["tokens"] * (2 * H * D + 8), "flops": 0}
    return {"bytes": case["rows"] * (2 * case["vocab"] + 20), "flops": 0}


def _ops_bytes(tokens, hidden, ffn):
    norm, rope_append, add_norm = 2 * hidden, 6 * hidden, 4 * hidden  # rope: q read + written, k and v read, two cache rows
    return 2 * (tokens * (norm + rope_append + add_norm + 3 * ffn) + 2 * hidden)


def tolerance(case):
    """About four times what the path differs by from the same computation in 64 bits on these inputs (measured: relative
    error 2.1e-4 to 3.7e-4 in fp16, 1.7e-3 to 3.0e-3 in bf16; largest single difference 1.5e-3 in fp16, 1.7e-2 in the fp16
    prefill, 2.5e-2 in bf16)."""
    if case["kind"] in ("move", "sample"):
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 1.2e-2, "max": 1e-1}
    return {"rel": 1.5e-3, "max": 7e-2 if case["kind"] == "prefill" else 6e-3}


# --------------------------------------------------------------------------- #
# what a program holds before the call
# --------------------------------------------------------------------------- #
def _dev():
    return torch.device("cuda")


def _randn(gen, shape, dtype, scale=1.0):
    t = torch.randn(shape, generator=gen, dtype=dtype, device=_dev())
    return t if scale == 1.0 else t.mul_(scale)


def _pools(gen, tokens, heads, head_dim, dtype):
    """K and V pools a quarter larger than the tokens in use, and the (permuted) slot of every token."""
    pool = tokens + tokens // 4 + 64
    slots = torch.randperm(pool, generator=gen, device=_dev())[:tokens].to(torch.int32)
    return _randn(gen, (pool, heads, head_dim), dtype), _randn(gen, (pool, heads, head_dim), dtype), slots


def _cuts(slots, lens):
    """The slot list cut into consecutive python lists of the given lengths."""
    flat, out, at = slots.tolist(), [], 0
    for n in lens:
        out.append(flat[at:at + n])
        at += n
    return out


def _padded(slots, lens):
    """Block table [B, width] and lengths of consecutive requests, on the device."""
    lens_t = torch.tensor(lens, dtype=torch.int64, device=_dev())
    width = max(lens)
    starts = torch.cumsum(lens_t, 0) - lens_t
    cols = torch.arange(width, device=_dev())
    at = torch.minimum(starts[:, None] + cols[None, :], torch.tensor(slots.numel() - 1, device=_dev()))
    table = torch.where(cols[None, :] < lens_t[:, None], slots[at], torch.zeros((), dtype=torch.int32, device=_dev()))
    return table.contiguous(), lens_t.to(torch.int32)


def _ops_state(gen, st, tokens, H, D, ffn, dtype, positions, scale=1.0):
    hidden = H * D
    st["x"] = _randn(gen, (tokens, hidden), dtype)
    st["delta"] = _randn(gen, (tokens, hidden), dtype, scale)  # what the layer adds to its residual stream
    st["residual"] = _randn(gen, (tokens, hidden), dtype)
    st["w1"], st["w2"] = _randn(gen, (hidden,), dtype), _randn(gen, (hidden,), dtype)
    st["qkv"] = _randn(gen, (tokens, 3 * hidden), dtype)       # q, k, v are column slices of the fused projection
    st["gate"], st["up"] = _randn(gen, (tokens, ffn), dtype), _randn(gen, (tokens, ffn), dtype)
    st["positions"] = torch.tensor(positions, dtype=torch.int64, device=_dev())
    st["cos_sin"] = mem.make_cos_sin_cache(max(positions) + 1, D, 10000.0, dtype, _dev())


def prepare(case, seed):
    kind, gen = case["kind"], torch.Generator(device=_dev()).manual_seed(seed)
    dtype, H, D = _DTYPES[case["dtype"]], case.get("heads", 0), case.get("head_dim", 0)
    st = {"kind": kind, "head_dim": D}
    if kind in ("layer", "decode"):
        groups = case.get("groups", 1)
        B = case["batch"] if kind == "layer" else groups * case["branches"]
        own = _between(case, B, case["own_lo"], case["own_hi"])
        st["k"], st["v"], slots = _pools(gen, groups * case["prefix"] + sum(own), H, D, dtype)
        lists = _cuts(slots, [case["prefix"]] * groups + own)
        st["prefix_lists"], st["own_lists"] = lists[:groups], lists[groups:]
        st["tables"] = kernels.DecodeTables.build(lists[:groups], [g * (B // groups) for g in range(groups + 1)],
                                                  lists[groups:], _dev(), num_heads=H, head_dim=D, dtype=dtype)
        if kind == "decode":
            st["q"] = _randn(gen, (B, H, D), dtype)
        else:  # the batch's new tokens take the last slot of every own list
            _ops_state(gen, st, B, H, D, case["ffn"], dtype, [case["prefix"] + n - 1 for n in own], scale=0.02)
            st["new_slots"] = torch.tensor([own_list[-1] for own_list in lists[groups:]], dtype=torch.int32, device=_dev())
    elif kind == "paged":
        B, G = case["branches"], case["kv_heads"]
        own = _between(case, B, case["own_lo"], case["own_hi"])
        st["k"], st["v"], slots = _pools(gen, case["prefix"] + sum(own), G, D, dtype)
        st["q"] = _randn(gen, (B, H, D), dtype)
        st["prefix"], st["prefix_table"] = case["prefix"], slots[:case["prefix"]].contiguous()
        st["table"], st["lens"] = _padded(slots[case["prefix"]:], own)
        st["head_mapping"] = torch.arange(G, dtype=torch.int32, device=_dev()).repeat_interleave(H // G)
    elif kind == "ragged":
        ctx = _contexts(case)
        st["k"], st["v"], slots = _pools(gen, sum(ctx), H, D, dtype)
        st["q"] = _randn(gen, (len(ctx), H, D), dtype)
        st["table"], st["lens"] = _padded(slots, ctx)
        st["head_mapping"] = torch.arange(H, dtype=torch.int32, device=_dev())
    elif kind == "prefill":
        new = _between(case, case["chunks"], case["new_lo"], case["new_hi"])
        ctx = [case["parent"] + n for n in new]
        st["k"], st["v"], slots = _pools(gen, sum(ctx), H, D, dtype)
        st["q"] = _randn(gen, (sum(new), H, D), dtype)
        st["new_lens"], st["contexts"] = new, _cuts(slots, ctx)
        st["tables"] = kernels.PrefillTables.build(new, st["contexts"], _dev())
    elif kind == "ops":
        T = case["tokens"]
        st["k"], st["v"], st["new_slots"] = _pools(gen, T, H, D, dtype)
        r = random.Random(case["lens"])
        _ops_state(gen, st, T, H, D, case["ffn"], dtype, [r.randrange(3072) for _ in range(T)])
    elif kind == "move":
        st["src"] = _randn(gen, (case["pool"], H, D), dtype)
        st["dst"] = torch.zeros((case["pool"], H, D), dtype=dtype, device=_dev())
        st["src_idx"] = torch.randperm(case["pool"], generator=gen, device=_dev())[:case["tokens"]]
        st["dst_idx"] = torch.randperm(case["pool"], generator=gen, device=_dev())[:case["tokens"]]
    else:
        rows = case["rows"]
        st["logits"] = _randn(gen, (rows, case["vocab"]), dtype, 4.0)
        st["temperature"] = torch.full((rows,), case["temperature"], device=_dev())
        st["top_p"] = torch.full((rows,), case["top_p"], device=_dev()) if case["top_p"] < 1.0 else None
        st["uniform"] = torch.rand(rows, generator=gen, device=_dev())
    return st


# --------------------------------------------------------------------------- #
# one pass
# --------------------------------------------------------------------------- #
def _layer_ops(st, attention):
    """A decoder layer's own kernels in their order, the projections between them left out."""
    D = st["head_dim"]
    T, hidden = st["x"].shape
    normed = kernels.vllm_rms_norm(st["x"], st["w1"], 1e-6)
    q, k, v = torch.chunk(st["qkv"], 3, dim=-1)
    kernels.rope_and_cache(st["positions"], q, k, v, st["cos_sin"], D, st["k"], st["v"], st["new_slots"],
                           key_in_place=False)
    out = {"normed": normed, "q": q, "k_cache": st["k"], "v_cache": st["v"]}
    if attention:
        out["attention"] = kernels.decode_attention(q.view(T, hidden // D, D), st["k"], st["v"], st["tables"])
    out["post_norm"] = kernels.fused_add_rms_norm(st["delta"], st["residual"], st["w2"], 1e-6)
    out["residual"] = st["residual"]
    out["activation"] = kernels.silu_mul(st["gate"], st["up"])
    return out


def run(st):
    kind = st["kind"]
    if kind in ("layer", "ops"):
        return _layer_ops(st, kind == "layer")
    if kind == "decode":
        return kernels.decode_attention(st["q"], st["k"], st["v"], st["tables"])
    if kind == "paged":
        return kernels.flash_paged_attention(st["q"], st["k"], st["v"], st["head_mapping"], st["prefix"],
                                             st["prefix_table"], st["lens"], st["table"])
    if kind == "ragged":
        return kernels.vllm_paged_attention(st["q"], st["k"], st["v"], st["head_mapping"], st["lens"], st["table"])
    if kind == "prefill":
        return kernels.prefill_attention(st["q"], st["k"], st["v"], st["tables"])
    if kind == "move":
        kernels.discontinuous_move_tokens(st["src"], st["dst"], st["src_idx"], st["dst_idx"])
        return st["dst"]
    return kernels.sample_top_p(st["logits"], st["temperature"], st["top_p"], st["uniform"])


# --------------------------------------------------------------------------- #
# the same outputs in 64 bits, by plain torch
# --------------------------------------------------------------------------- #
def _attend64(q, keys, values, causal_from=None, scores_at_once=1 << 28):
    """softmax(q k^T / sqrt(D)) v of `q` [n, H, D] over `keys`, `values` [m, G, D], query head h on KV head h * G // H.
    `causal_from`: query i sees the keys 0 to causal_from + i."""
    n, H, D = q.shape
    out = torch.empty((n, H, D), dtype=torch.float64, device=q.device)
    step = max(1, scores_at_once // keys.shape[0])
    for h in range(H):
        g = h * keys.shape[1] // H
        kt, v = keys[:, g].double().t().contiguous(), values[:, g].double()
        for at in range(0, n, step):
            s = (q[at:at + step, h].double() / math.sqrt(D)) @ kt
            if causal_from is not None:
                last = causal_from + at + torch.arange(s.shape[0], device=s.device)
                s.masked_fill_(torch.arange(s.shape[1], device=s.device)[None, :] > last[:, None], -math.inf)
            out[at:at + step, h] = torch.softmax(s, dim=-1) @ v
    return out


def _decode64(q, k, v, prefix_lists, own_lists):
    """Every request attends its group's prefix, then its own tokens; the groups hold equally many requests.  The requests
    of a group share one product with the prefix, and the two parts are joined by their log-sum-exp."""
    B, H, D = q.shape
    G, per = k.shape[1], B // max(1, len(prefix_lists))
    kv_head = torch.arange(H, device=q.device) * G // H
    out = torch.empty((B, H, D), dtype=torch.float64, device=q.device)
    q = q.double() / math.sqrt(D)

    def index(slots):
        return torch.as_tensor(slots, dtype=torch.int64, device=q.device)

    prefix_lse = torch.full((B, H), -math.inf, dtype=torch.float64, device=q.device)
    prefix_out = torch.zeros_like(out)
    for g, slots in enumerate(prefix_lists):
        rows = slice(g * per, (g + 1) * per)
        keys, values = k[index(slots)], v[index(slots)]
        for h in range(H):
            s = q[rows, h] @ keys[:, kv_head[h]].double().t().contiguous()
            prefix_lse[rows, h] = torch.logsumexp(s, dim=-1)
            prefix_out[rows, h] = torch.softmax(s, dim=-1) @ values[:, kv_head[h]].double()
    for b, slots in enumerate(own_lists):
        keys = k[index(slots)].double()[:, kv_head]
        s = (keys * q[b][None]).sum(-1)                                          # [n, H]
        lse = torch.logsumexp(s, dim=0)
        own = (torch.softmax(s, dim=0)[..., None] * v[index(slots)].double()[:, kv_head]).sum(0)
        both = torch.logaddexp(prefix_lse[b], lse)
        out[b] = torch.exp(prefix_lse[b] - both)[:, None] * prefix_out[b] + torch.exp(lse - both)[:, None] * own
    return out


def _layer64(st, attention):
    D, eps = st["head_dim"], 1e-6
    T, hidden = st["x"].shape

    def norm(x, w):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()

    q, k, v = (c.double().view(T, hidden // D, D) for c in torch.chunk(st["qkv"], 3, dim=-1))
    cos, sin = st["cos_sin"][st["positions"]].double()[:, None].chunk(2, dim=-1)

    def rotate(x):
        a, b = x.chunk(2, dim=-1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    q, slots = rotate(q), st["new_slots"].long()
    k_cache, v_cache = st["k"].double(), st["v"].double()
    k_cache[slots], v_cache[slots] = rotate(k), v
    out = {"normed": norm(st["x"].double(), st["w1"]), "q": q.reshape(T, hidden), "k_cache": k_cache, "v_cache": v_cache}
    if attention:
        out["attention"] = _decode64(q, k_cache, v_cache, st["prefix_lists"], st["own_lists"])
    residual, gate = st["residual"].double() + st["delta"].double(), st["gate"].double()
    out["post_norm"] = norm(residual, st["w2"])
    out["residual"] = residual
    out["activation"] = gate * torch.sigmoid(gate) * st["up"].double()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # whole numbers, drawn from a filter whose edge is a comparison of rounded sums
    st = prepare(case, seed)
    if kind in ("layer", "ops"):
        return _layer64(st, kind == "layer")
    if kind == "decode":
        return _decode64(st["q"], st["k"], st["v"], st["prefix_lists"], st["own_lists"])
    if kind in ("paged", "ragged"):
        own = [row[:n] for row, n in zip(st["table"].long(), st["lens"].tolist())]
        return _decode64(st["q"], st["k"], st["v"], [st["prefix_table"].long()] if kind == "paged" else [], own)
    if kind == "prefill":
        parts, at = [], 0
        for n, slots in zip(st["new_lens"], st["contexts"]):
            slots = torch.tensor(slots, dtype=torch.int64, device=_dev())
            parts.append(_attend64(st["q"][at:at + n], st["k"][slots], st["v"][slots], causal_from=len(slots) - n))
            at += n
        return torch.cat(parts)
    out = st["dst"].double()
    out[st["dst_idx"]] = st["src"][st["src_idx"]].double()
    return out
