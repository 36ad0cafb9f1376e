"""The workloads this package is timed on: the per-layer ops, attention and sampling of a forward
pass, called through the public entry points as a serving backend calls them.

A case names its family, the model dimensions and the batch; ``draw`` gives more cases of the same
ranges. Ragged lengths come from the case's own ``lens`` number, so the work of a case is known
without its inputs; values, page tables and token ids come from the seed given to ``prepare``.

Families:
  decode_layer  one layer of a decode step, op by op and eager (batches that have no captured
                graph): add + norm, q/k norm + RoPE + append, attention, add + norm, SiLU-and-mul
  decode_attn   the planned decode wrapper's run over a paged cache
  prefill       the planned prefill (or sink) wrapper's run, causal, ragged prompts
  step_mask     attention of one prefill step under custom masks: one plan, one run per layer
  verify        attention of a few drafted tokens per request over a long cached context, the
                tokens forming a tree (custom mask)
  block         the element-wise work of a prefill layer: embedding, add + norm, q/k norm + RoPE +
                append, gated activation
  sample        logits to tokens: safe_scaled_softmax, then a sampler
"""
from __future__ import annotations

import math
import random

import torch

from pie_amd import attention, ops, sampling

BF16 = torch.bfloat16
PAGE = 16
WORKSPACE = 128 << 20  # the float workspace Pie gives its wrappers
EPS = 1e-6
THETA = 1e6

# heads of one layer: query heads, kv heads, head dim
HEADS = {
    "llama8b": (32, 8, 128),   # and Qwen3-8B
    "llama1b": (32, 8, 64),
    "oss": (64, 8, 64),        # gpt-oss: attention sinks, every other layer in a window of 128
    "gemma": (16, 8, 256),
    "llama8b_tp4": (8, 2, 128),  # one rank's heads under four-way tensor parallelism
}
HIDDEN = {"llama8b": (4096, 14336, 128256), "qwen8b": (4096, 12288, 151936), "llama1b": (2048, 8192, 128256)}


def listed():
    return [
        # one sequence decoding alone: latency and launches
        {"name": "decode_layer_1", "family": "decode_layer", "batch": 1, "lo": 900, "hi": 1100, "lens": 1},
        # an ordinary decode batch, odd in size
        {"name": "decode_layer_45", "family": "decode_layer", "batch": 45, "lo": 128, "hi": 2048, "lens": 2},
        # a full decode batch over mixed contexts (Qwen3-8B, contexts U[128, 4096])
        {"name": "decode_attn_256", "family": "decode_attn", "model": "llama8b", "batch": 256, "lo": 128, "hi": 4096,
         "lens": 3},
        # a few long conversations or documents
        {"name": "decode_attn_long", "family": "decode_attn", "model": "llama8b", "batch": 3, "lo": 16000, "hi": 32000,
         "lens": 4},
        # 64 fresh prompts of U[1, 2048] tokens (Llama-3-8B): the largest case
        {"name": "prefill_64", "family": "prefill", "model": "llama8b", "batch": 64, "lo": 1, "hi": 2048, "ctx": 0,
         "lens": 5},
        # gpt-oss: a full layer and a windowed one, with sinks
        {"name": "prefill_oss", "family": "prefill", "model": "oss", "batch": 12, "lo": 64, "hi": 2048, "ctx": 0,
         "lens": 6},
        # Gemma heads; chunks of prompts that continue a cached prefix
        {"name": "prefill_gemma", "family": "prefill", "model": "gemma", "batch": 7, "lo": 100, "hi": 2000, "ctx": 1000,
         "lens": 7},
        # a Llama-3.2-1B step as Pie runs it: masks always given, planned once, 16 layers
        {"name": "step_mask", "family": "step_mask", "model": "llama1b", "batch": 6, "lo": 16, "hi": 1200, "ctx": 300,
         "layers": 16, "lens": 8},
        # speculative decoding: a tree of drafted tokens per request verified over its context
        {"name": "verify_tree", "family": "verify", "model": "llama8b", "batch": 4, "qo": 13, "lo": 1000, "hi": 9000,
         "lens": 9},
        # a prefill layer's element-wise work (Qwen3-8B, 8192 tokens)
        {"name": "block_8192", "family": "block", "model": "qwen8b", "tokens": 8192, "lens": 10},
        # an ordinary sampling step: a few rows, nucleus sampling, bf16 logits
        {"name": "sample_9", "family": "sample", "rows": 9, "vocab": 151936, "dtype": "bf16", "sampler": "top_p"},
        # the full decode batch's sampling step, top-k and top-p per row, fp32 logits
        {"name": "sample_256", "family": "sample", "rows": 256, "vocab": 128256, "dtype": "fp32",
         "sampler": "top_k_top_p"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    lens = rng.randrange(1 << 20)
    family = rng.choice(["decode_layer", "decode_attn", "decode_attn", "prefill", "prefill", "step_mask", "verify",
                         "block", "sample", "sample"])
    if family == "decode_layer":
        return {"family": family, "batch": _log(rng, 1, 64), "lo": 64, "hi": _log(rng, 256, 4096), "lens": lens}
    if family == "decode_attn":
        batch = _log(rng, 1, 256)
        hi = _log(rng, 256, min(32000, 1000000 // batch))
        return {"family": family, "model": rng.choice(["llama8b", "llama8b", "oss", "gemma", "llama8b_tp4"]),
                "batch": batch, "lo": max(1, int(hi * rng.choice([0.03, 0.5]))), "hi": hi, "lens": lens}
    if family == "prefill":
        batch = _log(rng, 1, 32)
        hi = _log(rng, 64, min(6000, 30000 // batch))
        return {"family": family, "model": rng.choice(["llama8b", "llama8b", "oss", "gemma", "llama8b_tp4"]),
                "batch": batch, "lo": rng.randint(1, hi), "hi": hi, "ctx": rng.choice([0, 0, _log(rng, 50, 2000)]),
                "lens": lens}
    if family == "step_mask":
        batch = _log(rng, 1, 12)
        hi = _log(rng, 32, 4000 // batch)
        return {"family": family, "model": rng.choice(["llama1b", "llama8b"]), "batch": batch, "lo": rng.randint(1, hi),
                "hi": hi, "ctx": rng.choice([0, _log(rng, 20, 1000)]), "layers": 16, "lens": lens}
    if family == "verify":
        return {"family": family, "model": rng.choice(["llama8b", "llama1b", "llama8b_tp4"]),
                "batch": _log(rng, 1, 16), "qo": rng.randint(2, 40), "lo": 200, "hi": _log(rng, 500, 12000),
                "lens": lens}
    if family == "block":
        return {"family": family, "model": rng.choice(["llama8b", "qwen8b", "llama1b"]), "tokens": _log(rng, 16, 8192),
                "lens": lens}
    return {"family": family, "rows": _log(rng, 1, 256), "vocab": rng.choice([32000, 128256, 151936, 201088, 100277]),
            "dtype": rng.choice(["bf16", "fp32"]),
            "sampler": rng.choice(["top_p", "top_k_top_p", "top_k", "min_p", "plain"])}


# ------------------------------------------------------------------------------- batches
def _lens(case):
    """(cached tokens before the call, new tokens) of each request."""
    r = random.Random(case["lens"])
    family, n = case["family"], case.get("batch")
    if family in ("decode_layer", "decode_attn"):
        return [r.randint(case["lo"], case["hi"]) - 1 for _ in range(n)], [1] * n
    if family == "verify":
        return [r.randint(case["lo"], case["hi"]) for _ in range(n)], [case["qo"]] * n
    new = [r.randint(case["lo"], case["hi"]) for _ in range(n)]
    return [r.randint(case["ctx"] // 2, case["ctx"]) for _ in range(n)], new


def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(seed * 64 + what)


def _randn(shape, g, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=BF16).mul_(std).add_(mean)


def _tables(ctx, new, seed):
    """Page tables over a randomly permuted pool, on the device as Pie keeps them."""
    total = [c + n for c, n in zip(ctx, new)]
    pages = [-(-t // PAGE) for t in total]
    cum = lambda xs: torch.tensor([sum(xs[:i]) for i in range(len(xs) + 1)], dtype=torch.int32, device="cuda")
    n = sum(pages)
    bidx = [b for b, k in enumerate(new) for _ in range(k)]
    pos = [c + i for c, k in zip(ctx, new) for i in range(k)]
    i32 = lambda xs: torch.tensor(xs, dtype=torch.int32, device="cuda")
    return {"qo_indptr": cum(new), "kv_indptr": cum(pages), "pages": n,
            "kv_indices": torch.randperm(n, generator=_gen(seed, 40), device="cuda").to(torch.int32),
            "last": i32([t - PAGE * (p - 1) for t, p in zip(total, pages)]), "total": total,
            "bidx": i32(bidx), "pos": i32(pos)}


def _tree_masks(ctx, qo, seed):
    """Per request a flattened [qo, ctx + qo] mask: the context, the token itself and its
    ancestors in a random tree of drafted tokens."""
    r = random.Random(seed)
    parts = []
    for c in ctx:
        tree = torch.zeros((qo, qo), dtype=torch.bool)
        for i in range(qo):
            if i:
                tree[i] = tree[r.randrange(i)]
            tree[i, i] = True
        parts.append(torch.cat([torch.ones((qo, c), dtype=torch.bool), tree], 1).flatten())
    return torch.cat(parts).cuda()


def _causal_masks(ctx, new):
    parts = []
    for c, n in zip(ctx, new):
        t = torch.arange(c + n, device="cuda")
        parts.append((t[None, :] <= c + torch.arange(n, device="cuda")[:, None]).flatten())
    return torch.cat(parts)


def _decode_wrapper(t, heads, ws):
    w = attention.BatchDecodeWithPagedKVCacheWrapper(ws, "NHD")
    w.plan(t["kv_indptr"], t["kv_indices"], t["last"], *heads, PAGE, q_data_type=BF16)
    return w


def _windows(case):
    """The layers of one pass: gpt-oss alternates full attention and a window of 128 tokens."""
    return [-1, 127] if case.get("model") == "oss" else [-1]


def prepare(case, seed):
    family = case["family"]
    s = {"case": case}
    if family == "sample":
        B, V = case["rows"], case["vocab"]
        # rows of different sharpness, as a model's confident and unsure steps give
        spread = torch.rand((B, 1), generator=_gen(seed, 1), device="cuda") * 3 + 2
        logits = torch.randn((B, V), generator=_gen(seed, 2), device="cuda").mul_(spread)
        s["logits"] = logits.to(BF16) if case["dtype"] == "bf16" else logits
        u = lambda k: torch.rand(B, generator=_gen(seed, k), device="cuda")
        s["temps"], s["top_p"], s["min_p"] = 0.6 + 0.6 * u(3), 0.8 + 0.19 * u(4), 0.02 + 0.1 * u(5)
        s["top_k"] = (20 + 40 * u(6)).to(torch.int32)
        s["seed"] = seed
        return s
    if family == "block":
        T, (H, I, V) = case["tokens"], HIDDEN[case["model"]]
        Hq, Hkv, D = HEADS["llama1b" if case["model"] == "llama1b" else "llama8b"]
        ids = torch.randint(0, V, (T,), generator=_gen(seed, 1), device="cuda").to(torch.int32)
        s.update(ids=ids, table=_randn((V, H), _gen(seed, 2), 0.5), o=_randn((T, H), _gen(seed, 3)),
                 w=_randn((H,), _gen(seed, 4), 0.1, 1.0), gate_up=_randn((T, 2 * I), _gen(seed, 5), 1.4))
        r = random.Random(case["lens"])
        new = []
        while sum(new) < T:  # the prompts of the step
            new.append(min(T - sum(new), r.randint(1, 2048)))
        t = _tables([0] * len(new), new, seed)
    else:
        ctx, new = _lens(case)
        T = sum(new)
        Hq, Hkv, D = HEADS[case.get("model", "llama8b")]
        t = _tables(ctx, new, seed)
    s.update(t=t, heads=(Hq, Hkv, D))
    layers = case.get("layers", len(_windows(case)))
    s["caches"] = [_randn((t["pages"], 2, PAGE, Hkv, D), _gen(seed, 10 + i)) for i in range(layers)]
    if family in ("block", "decode_layer"):
        s["qkv"] = _randn((T, (Hq + 2 * Hkv) * D), _gen(seed, 6))
        s["qw"], s["kw"] = _randn((D,), _gen(seed, 7), 0.1, 1.0), _randn((D,), _gen(seed, 8), 0.1, 1.0)
        if family == "block":
            return s
        H, I, _ = HIDDEN["qwen8b"]
        s.update(down=_randn((T, H), _gen(seed, 50)), residual=_randn((T, H), _gen(seed, 51)),
                 o=_randn((T, H), _gen(seed, 52)), w1=_randn((H,), _gen(seed, 53), 0.1, 1.0),
                 w2=_randn((H,), _gen(seed, 54), 0.1, 1.0), gate_up=_randn((T, 2 * I), _gen(seed, 55), 1.4))
    s["ws"] = torch.zeros(WORKSPACE, dtype=torch.uint8, device="cuda")
    if family == "decode_layer":
        s["wrapper"] = _decode_wrapper(t, s["heads"], s["ws"])
        return s
    s["q"] = [_randn((T, Hq, D), _gen(seed, 30 + i)) for i in range(layers)]
    if case["model"] == "oss":
        s["sinks"] = torch.randn(Hq, generator=_gen(seed, 60), device="cuda")
        s["wrappers"] = []
        for window in _windows(case):
            ws = torch.zeros(WORKSPACE, dtype=torch.uint8, device="cuda")
            w = attention.BatchAttentionWithAttentionSinkWrapper(ws, "NHD", window_left=window, q_data_type=BF16,
                                                                 head_dim_qk=D, head_dim_vo=D)
            w.plan(t["qo_indptr"], t["kv_indptr"], t["kv_indices"], t["last"], Hq, Hkv, D, PAGE)
            s["wrappers"].append(w)
        return s
    if family == "decode_attn":
        s["wrapper"] = _decode_wrapper(t, s["heads"], s["ws"])
        return s
    s["wrapper"] = attention.BatchPrefillWithPagedKVCacheWrapper(s["ws"], "NHD")
    if family == "prefill":
        _plan_prefill(s, causal=True)
    elif family == "verify":
        s["mask"] = _tree_masks(ctx, case["qo"], seed)
        _plan_prefill(s, custom_mask=s["mask"])
    else:
        s["mask"] = _causal_masks(ctx, new)
    return s


def _plan_prefill(s, **visible):
    t = s["t"]
    s["wrapper"].plan(t["qo_indptr"], t["kv_indptr"], t["kv_indices"], t["last"], *s["heads"], PAGE, q_data_type=BF16,
                      **visible)


def _prologue(s):
    Hq, Hkv, D = s["heads"]
    t, T = s["t"], s["qkv"].shape[0]
    q, k, v = torch.split(s["qkv"], [Hq * D, Hkv * D, Hkv * D], dim=-1)
    return ops.qk_rms_norm_rope_append(q.view(T, Hq, D), k.view(T, Hkv, D), v.view(T, Hkv, D), s["qw"], s["kw"], EPS,
                                       t["pos"], t["bidx"], t["pos"], s["caches"][0], t["kv_indices"], t["kv_indptr"],
                                       t["last"], rope_theta=THETA)


def run(state):
    s, family = state, state["case"]["family"]
    if family == "decode_layer":
        normed, residual = ops.add_rms_norm(s["down"], s["residual"], s["w1"], EPS)
        q, k = _prologue(s)
        attn = s["wrapper"].run(q, s["caches"][0])
        normed2, residual2 = ops.add_rms_norm(s["o"], residual, s["w2"], EPS)
        act = ops.silu_and_mul(s["gate_up"])
        return [normed, residual, q, k, attn, normed2, residual2, act, s["caches"][0]]
    if family == "block":
        hidden = ops.embedding(s["ids"], s["table"])
        normed, residual = ops.add_rms_norm(s["o"], hidden, s["w"], EPS)
        q, k = _prologue(s)
        act = ops.silu_and_mul(s["gate_up"])
        return [hidden, normed, residual, q, k, act, s["caches"][0]]
    if family == "sample":
        probs = sampling.safe_scaled_softmax(s["logits"], s["temps"])
        p, mode, kw = probs.float(), s["case"]["sampler"], {"seed": s["seed"], "offset": 0}
        if mode == "top_p":
            token = sampling.top_p_sampling_from_probs(p, s["top_p"], **kw)
        elif mode == "top_k":
            token = sampling.top_k_sampling_from_probs(p, s["top_k"], **kw)
        elif mode == "min_p":
            token = sampling.min_p_sampling_from_probs(p, s["min_p"], **kw)
        elif mode == "plain":
            token = sampling.sampling_from_probs(p, **kw)
        else:
            token = sampling.top_k_top_p_sampling_from_probs(p, s["top_k"], s["top_p"], **kw)
        return [probs, token]
    if s["case"]["model"] == "oss":
        return [w.run(q, c, s["sinks"]) for w, q, c in zip(s["wrappers"], s["q"], s["caches"])]
    if family == "step_mask":
        _plan_prefill(s, custom_mask=s["mask"])
        return [s["wrapper"].run(q, c) for q, c in zip(s["q"], s["caches"])]
    return [s["wrapper"].run(s["q"][0], s["caches"][0])]


# ------------------------------------------------------------------------------- work, tolerance
def _attention_work(ctx, new, heads, window=-1, tree=False):
    Hq, Hkv, D = heads
    pairs = seen = 0
    for c, n in zip(ctx, new):
        first = 0 if window < 0 else max(0, c - window)  # oldest position any new token sees
        seen += c + n - first
        if tree:
            pairs += n * c + n * (n + 1) // 2
        else:
            pairs += sum(min(c + i + 1, window + 1) if window >= 0 else c + i + 1 for i in range(n))
    return {"bytes": 4 * sum(new) * Hq * D + 4 * seen * Hkv * D, "flops": 4 * pairs * Hq * D}


def work(case):
    family = case["family"]
    if family == "sample":
        size = 2 if case["dtype"] == "bf16" else 4
        n = case["rows"] * case["vocab"]
        return {"bytes": 2 * size * n, "flops": 5 * n}
    if family == "block":
        T, (H, I, _) = case["tokens"], HIDDEN[case["model"]]
        Hq, Hkv, D = HEADS["llama1b" if case["model"] == "llama1b" else "llama8b"]
        return {"bytes": 2 * T * (2 * H + 3 * H + (2 * Hq + 5 * Hkv) * D + 3 * I), "flops": T * (6 * H + 10 * Hq * D + 6 * I)}
    ctx, new = _lens(case)
    heads = HEADS[case.get("model", "llama8b")]
    if family == "decode_layer":
        w = _attention_work(ctx, new, heads)
        H, I, _ = HIDDEN["qwen8b"]
        T, (Hq, Hkv, D) = sum(new), heads
        w["bytes"] += 2 * T * (7 * H + (2 * Hq + 4 * Hkv) * D + 3 * I)
        w["flops"] += T * (12 * H + 10 * Hq * D + 6 * I)
        return w
    parts = [_attention_work(ctx, new, heads, w, family == "verify") for w in _windows(case)] * (case.get("layers", 1))
    total = {k: sum(p[k] for p in parts) for k in parts[0]}
    if family == "step_mask":
        total["bytes"] += sum((c + n) * n for c, n in zip(ctx, new))
    return total


def tolerance(case):
    family = case["family"]
    if family == "sample":
        # fp32 sums over the vocabulary in another order; bf16 probabilities may round the other way
        return {"rel": 2e-3 if case["dtype"] == "bf16" else 1e-5, "differ": 0.005}
    if family == "block":
        return {"rel": 2e-3, "max": 0.02}
    # bf16 outputs of softmax-weighted sums whose weights are rounded to bf16
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------------------- 64-bit results
def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos):
    D = x.shape[-1]
    inv = THETA ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    a = pos.double()[:, None, None] * inv
    lo, hi = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([lo * a.cos() - hi * a.sin(), lo * a.sin() + hi * a.cos()], -1)


def _prologue64(s):
    """q, k and the cache after the append."""
    Hq, Hkv, D = s["heads"]
    t, T = s["t"], s["qkv"].shape[0]
    x = s["qkv"].double().view(T, Hq + 2 * Hkv, D)
    q = _rope64(_norm64(x[:, :Hq], s["qw"]), t["pos"])
    k = _rope64(_norm64(x[:, Hq:Hq + Hkv], s["kw"]), t["pos"])
    cache = s["caches"][0].double()
    pos, b = t["pos"].long(), t["bidx"].long()
    page = t["kv_indices"].long()[t["kv_indptr"].long()[b] + pos // PAGE]
    cache[page, 0, pos % PAGE] = k
    cache[page, 1, pos % PAGE] = x[:, Hq + Hkv:]
    return q, k, cache


def _attention64(s, q, cache, window=-1, sinks=None, masks=None):
    Hq, Hkv, D = s["heads"]
    t, G = s["t"], Hq // Hkv
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    qi, ki, at = t["qo_indptr"].tolist(), t["kv_indptr"].tolist(), 0
    for b, total in enumerate(t["total"]):
        n = qi[b + 1] - qi[b]
        kv = cache[t["kv_indices"][ki[b]:ki[b + 1]].long()].double().transpose(0, 1)
        kv = kv.reshape(2, -1, Hkv, D)[:, :total]
        i = torch.arange(n, device="cuda")[:, None] + total - n
        j = torch.arange(total, device="cuda")[None, :]
        if masks is not None:
            see = masks[at:at + n * total].view(n, total)
            at += n * total
        else:
            see = (j <= i) & ((j >= i - window) if window >= 0 else True)
        for h in range(Hq):
            sc = q[qi[b]:qi[b + 1], h].double() @ kv[0, :, h // G].t().contiguous() / math.sqrt(D)
            sc = sc.masked_fill(~see, -math.inf)
            if sinks is not None:
                sc = torch.cat([sc, sinks[h].double().expand(n, 1)], 1)
            p = torch.softmax(sc, -1)[:, :total]
            out[qi[b]:qi[b + 1], h] = p @ kv[1, :, h // G].contiguous()
    return out


def exact(case, seed):
    family = case["family"]
    s = prepare(case, seed)
    if family == "sample":
        return [torch.softmax(s["logits"].double() / s["temps"].double()[:, None], -1), None]
    silu = lambda x: torch.nn.functional.silu(x[:, : x.shape[1] // 2].double()) * x[:, x.shape[1] // 2:].double()
    if family == "block":
        hidden = s["table"][s["ids"].long()].double()
        residual = s["o"].double() + hidden
        q, k, cache = _prologue64(s)
        return [hidden, _norm64(residual, s["w"]), residual, q, k, silu(s["gate_up"]), cache]
    if family == "decode_layer":
        residual = s["down"].double() + s["residual"].double()
        q, k, cache = _prologue64(s)
        residual2 = s["o"].double() + residual
        return [_norm64(residual, s["w1"]), residual, q, k, _attention64(s, q, cache), _norm64(residual2, s["w2"]),
                residual2, silu(s["gate_up"]), cache]
    return [_attention64(s, q, c, w, s.get("sinks"), s.get("mask"))
            for q, c, w in zip(s["q"], s["caches"], _windows(case) * len(s["q"]))]
