"""The work that serving has this framework do, as cases that can be timed and checked.

Five paths, each at the sizes that the presets of ``ome_amd.models.config`` give it:

* ``llama``: one step of the Llama-3-8B runtime through ``ModelRunner.launch`` (all 32 layers, paged KV
  cache, HIP-graph decode), decode rows alone or beside a chunk of prompts, bf16 or fp8 KV cache;
* ``moe``: routing and experts of one mixture-of-experts layer (``ops.moe_route`` + ``ops.fused_moe``),
  bf16 experts, or fp8 experts with 128 x 128 block scales;
* ``mla``: attention of one multi-head-latent layer over the paged latent cache (``ops.mla_attn``), decode
  rows and prompt rows;
* ``gdn``: the gated delta rule of one Qwen3-Next layer between its two projections (short convolution,
  scan, gated norm), prompts and decode rows;
* ``mamba``: the same of one Nemotron-H Mamba-2 layer.

Sizes of a case follow from the case alone, values from the seed.
"""
import math
import random

import torch

from ome_amd import ops
from ome_amd.models.config import preset
from ome_amd.models.quant import Fp8Experts
from ome_amd.runtime.model_runner import ModelRunner, default_buckets
from ome_amd.runtime.request import Request, SamplingParams
from ome_amd.runtime.scheduler import ScheduledChunk, StepBatch

DEV = "cuda"
PAGE = 16

# Llama-3-8B (preset "llama-3-8b")
HID, LAYERS, HQ, HKV, HD, FF, VOCAB, THETA, EPS = 4096, 32, 32, 8, 128, 14336, 128256, 500000.0, 1e-5

# experts, chosen, width, expert width, router, gated
MOE = {
    "mixtral-8x7b": (8, 2, 4096, 14336, "softmax", True),
    "qwen3-next-80b-a3b": (512, 10, 2048, 512, "softmax", True),
    "deepseek-v3": (256, 8, 7168, 2048, "groups", True),
    "nemotron-3-nano-30b-a3b": (128, 6, 2688, 1856, "sigmoid", False),
}


def listed():
    return [
        # one chat user: a decode step of a single request at ~700 tokens of context
        {"name": "llama_decode_1", "kind": "llama", "decodes": 1, "ctx": 700, "prompts": 0, "prompt_tokens": 0, "past": 0, "fp8_kv": False},
        # the benchmark's steady state: 256 requests with ragged contexts of N(480,240)/(300,150) lengths
        {"name": "llama_decode_256", "kind": "llama", "decodes": 256, "ctx": 630, "prompts": 0, "prompt_tokens": 0, "past": 0, "fp8_kv": False},
        # its other step: the chunk budget filled with new prompts while the running requests decode
        {"name": "llama_mixed_2048", "kind": "llama", "decodes": 200, "ctx": 630, "prompts": 5, "prompt_tokens": 2048, "past": 0, "fp8_kv": False},
        # a long document in chunks: the last 1500 tokens of a prompt of about 7600, few decodes beside it, fp8 cache
        {"name": "llama_chunk_long_fp8kv", "kind": "llama", "decodes": 17, "ctx": 1900, "prompts": 1, "prompt_tokens": 1500, "past": 6100, "fp8_kv": True},
        # decode steps of a many-expert layer: nearly every expert has a few rows, weights dominate
        {"name": "moe_decode", "kind": "moe", "model": "qwen3-next-80b-a3b", "tokens": 48, "fp8": False},
        # a prompt chunk through few large experts
        {"name": "moe_prefill", "kind": "moe", "model": "mixtral-8x7b", "tokens": 3000, "fp8": False},
        # fp8 block-scaled experts at a mixed step's row count
        {"name": "moe_fp8", "kind": "moe", "model": "deepseek-v3", "tokens": 700, "fp8": True},
        # DeepSeek-V3 decode, all 128 heads on one GPU, ragged contexts
        {"name": "mla_decode", "kind": "mla", "seqs": 48, "rows": 1, "ctx": 3000, "heads": 128},
        # DeepSeek-V2-Lite / an eighth of DeepSeek-V3's heads: prompts
        {"name": "mla_prefill", "kind": "mla", "seqs": 3, "rows": 1300, "ctx": 1300, "heads": 16},
        # Qwen3-Next prompts: a chunk of three
        {"name": "gdn_prefill", "kind": "gdn", "seqs": 3, "tokens": 4000, "shards": 1},
        # Qwen3-Next decode
        {"name": "gdn_decode", "kind": "gdn", "seqs": 64, "tokens": 64, "shards": 1},
        # Nemotron-H prompts
        {"name": "mamba_prefill", "kind": "mamba", "seqs": 4, "tokens": 3500, "shards": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["llama", "moe", "moe", "mla", "mla", "gdn", "gdn", "mamba"])
    if kind == "llama":
        ctx = _log(rng, 64, 3000)
        decodes = min(_log(rng, 1, 256), 160000 // ctx)
        if rng.random() < 0.5:
            return {"kind": kind, "decodes": decodes, "ctx": ctx, "prompts": 0, "prompt_tokens": 0, "past": 0, "fp8_kv": rng.random() < 0.3}
        tokens = _log(rng, 40, 2000)
        prompts = max(1, min(_log(rng, 1, 8), tokens // 20))
        return {"kind": kind, "decodes": min(decodes, 200), "ctx": ctx, "prompts": prompts, "prompt_tokens": tokens,
                "past": rng.choice([0, 0, _log(rng, 16, 6000 // prompts)]), "fp8_kv": rng.random() < 0.3}
    if kind == "moe":
        model = rng.choice(sorted(MOE))
        fp8 = model == "deepseek-v3"   # its experts are published in fp8; the others are served in bf16
        return {"kind": kind, "model": model, "tokens": _log(rng, 1, 1000 if fp8 else 3000), "fp8": fp8}
    if kind == "mla":
        heads = rng.choice([16, 16, 32, 64, 128])
        if rng.random() < 0.5:
            seqs = _log(rng, 1, 128)
            return {"kind": kind, "seqs": seqs, "rows": 1, "ctx": _log(rng, 64, min(8000, 400000 // seqs)), "heads": heads}
        rows = _log(rng, 20, 4000 * 16 // heads)
        past = rng.choice([0, 0, _log(rng, 16, 3000)])
        seqs = max(1, min(_log(rng, 1, 8), 6000 * 16 // heads // rows))
        return {"kind": kind, "seqs": seqs, "rows": rows, "ctx": rows + past, "heads": heads}
    shards = rng.choice([1, 1, 2, 4])
    if rng.random() < 0.4:
        n = _log(rng, 2, 256)
        return {"kind": kind, "seqs": n, "tokens": n, "shards": shards}
    tokens = _log(rng, 30, 8000)
    return {"kind": kind, "seqs": max(1, min(_log(rng, 1, 16), tokens // 8)), "tokens": tokens, "shards": shards}


# ------------------------------------------------------------------ sizes and values
def _lens(case, tag, n, mean, least=1):
    """n ragged lengths around ``mean`` (a quarter to seven quarters of it), from the case alone."""
    r = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")) + tag)
    return [max(least, int(mean * r.uniform(0.25, 1.75))) for _ in range(n)]


def _parts(case, tag, n, total):
    """``total`` in n ragged parts of at least 1."""
    w = _lens(case, tag, n, 1000)
    cut = [total * sum(w[:i]) // sum(w) for i in range(n + 1)]
    out = [max(1, b - a) for a, b in zip(cut, cut[1:])]
    out[out.index(max(out))] += total - sum(out)
    return out


def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + sum(ord(c) * 257 ** (i % 5) for i, c in enumerate(tag))) % (1 << 62))
    return g


def _normal(seed, tag, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    return torch.empty(*shape, dtype=dtype, device=DEV).normal_(mean, std, generator=_gen(seed, tag))


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# ------------------------------------------------------------------ Llama-3-8B steps
def _llama_weights(seed):
    """The checkpoint, tensor by tensor, in the published layout."""
    deep = 0.02 / math.sqrt(2 * LAYERS)
    yield "model.embed_tokens.weight", _normal(seed, "embed", VOCAB, HID)
    yield "model.norm.weight", _normal(seed, "norm", HID, std=0.1, mean=1.0)
    yield "lm_head.weight", _normal(seed, "head", VOCAB, HID, std=0.02)
    for i in range(LAYERS):
        yield from _llama_layer(seed, i, deep)


def _llama_layer(seed, i, deep=0.02 / math.sqrt(2 * LAYERS)):
    p = "model.layers.%d." % i
    for name, shape, std in (("self_attn.q_proj", (HQ * HD, HID), 0.02), ("self_attn.k_proj", (HKV * HD, HID), 0.02),
                             ("self_attn.v_proj", (HKV * HD, HID), 0.02), ("self_attn.o_proj", (HID, HQ * HD), deep),
                             ("mlp.gate_proj", (FF, HID), 0.02), ("mlp.up_proj", (FF, HID), 0.02),
                             ("mlp.down_proj", (HID, FF), deep)):
        yield p + name + ".weight", _normal(seed, p + name, *shape, std=std)
    for name in ("input_layernorm", "post_attention_layernorm"):
        yield p + name + ".weight", _normal(seed, p + name, HID, std=0.1, mean=1.0)


def _llama_sizes(case):
    """[(cached tokens, tokens of this step)] of every request: the prompts, then the decodes."""
    new = _parts(case, "p", case["prompts"], case["prompt_tokens"]) if case["prompts"] else []
    return [(case["past"], n) for n in new] + [(n - 1, 1) for n in _lens(case, "d", case["decodes"], case["ctx"], 2)]


def _llama_past(seed, layer, n, fp8):
    """Cached keys and values of ``n`` tokens (for an fp8 cache: values that it holds as they are)."""
    kv = [_normal(seed, "past%d%s" % (layer, x), n, HKV, HD) for x in "kv"]
    return [x.to(torch.float8_e4m3fn).to(torch.bfloat16) for x in kv] if fp8 else kv


def _llama_tokens(seed, sizes):
    g = torch.Generator()
    g.manual_seed(int(seed) + 17)
    return torch.randint(3, VOCAB, (sum(n for _, n in sizes),), generator=g)


def _llama_prepare(case, seed):
    sizes = _llama_sizes(case)
    longest = max(a + n for a, n in sizes)
    context = max(4096, -(-longest // 1024) * 1024)
    bucket = next(b for b in default_buckets(256) if b >= max(1, case["decodes"]))
    total = sum(-(-(a + n) // PAGE) * PAGE for a, n in sizes)
    runner = ModelRunner(preset("llama-3-8b"), device=DEV, max_running=256, max_context=context, max_total_tokens=total + 2 * context,
                         cuda_graph=False, cuda_graph_bs=[bucket], kv_cache_dtype_name="fp8" if case["fp8_kv"] else "auto", keep_logits=True)
    runner.model.load_hf_weights(_llama_weights(seed))
    free = torch.randperm(runner.pages.num_pages - 1, generator=torch.Generator().manual_seed(int(seed))) + 1   # pages of a pool in use
    tokens = _llama_tokens(seed, sizes).tolist()
    chunks, slots, p, t = [], [], 0, 0
    for a, n in sizes:
        pages = free[p:p + -(-(a + n) // PAGE)]
        p += len(pages)
        at = torch.arange(a)
        slots.append(pages[at // PAGE] * PAGE + at % PAGE)
        r = Request([0] * a + tokens[t:t + n], SamplingParams(ignore_eos=True))
        t += n
        r.pages, r.req_slot, r.num_cached = pages.tolist(), runner.slots.alloc(), a
        runner.slots.set_pages(r.req_slot, 0, r.pages)
        chunks.append(ScheduledChunk(r, a, n, True, want=[n - 1]))
    runner.slots.flush()
    slots = torch.cat(slots).to(device=DEV, dtype=torch.int32)
    for i in range(LAYERS):
        if slots.numel():
            k, v = _llama_past(seed, i, slots.numel(), case["fp8_kv"])
            ops.kv_cache_write(k, v, *runner.kv.layer(i), slots)
    mode = "decode"
    if case["prompts"]:
        mode = "mixed" if case["decodes"] else "prefill"
    else:
        runner.use_graph = True
        runner.capture_graphs()
    return {"kind": "llama", "runner": runner, "batch": StepBatch(mode, chunks)}


def _llama_run(s):
    return {"logits": s["runner"].launch(s["batch"]).logits}


def _llama_exact(case, seed):
    sizes = _llama_sizes(case)
    past = [a for a, _ in sizes]
    new = [n for _, n in sizes]
    rows = torch.cat([torch.arange(a, a + n) for a, n in sizes]).to(DEV)
    inv = 1.0 / THETA ** (torch.arange(0, HD, 2, dtype=torch.float64, device=DEV) / HD)
    ang = rows[:, None].double() * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(x):
        a, b = x[..., :HD // 2], x[..., HD // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def norm(x, w):
        return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()

    x = _normal(seed, "embed", VOCAB, HID)[_llama_tokens(seed, sizes).to(DEV)].double()
    for i in range(LAYERS):
        w = {k.split(".", 3)[3].rsplit(".", 1)[0]: v for k, v in _llama_layer(seed, i)}
        h = norm(x, w["input_layernorm"])
        q, k, v = ((h @ w["self_attn." + m].double().T).view(len(h), -1, HD) for m in ("q_proj", "k_proj", "v_proj"))
        q, k = rope(q), rope(k)
        pk, pv = _llama_past(seed, i, sum(past), case["fp8_kv"]) if sum(past) else (k[:0], v[:0])
        o, a0, n0 = torch.empty_like(q), 0, 0
        for a, n in zip(past, new):
            kk = torch.cat([pk[a0:a0 + a].double(), k[n0:n0 + n]]).repeat_interleave(HQ // HKV, 1).transpose(0, 1)
            vv = torch.cat([pv[a0:a0 + a].double(), v[n0:n0 + n]]).repeat_interleave(HQ // HKV, 1).transpose(0, 1)
            sc = q[n0:n0 + n].transpose(0, 1) @ kk.transpose(1, 2).contiguous() / math.sqrt(HD)
            if n > 1:
                sc.masked_fill_(torch.ones(n, a + n, dtype=torch.bool, device=DEV).triu(a + 1), -math.inf)
            o[n0:n0 + n] = (sc.softmax(-1) @ vv).transpose(0, 1)
            a0, n0 = a0 + a, n0 + n
        x = x + o.reshape(len(h), -1) @ w["self_attn.o_proj"].double().T
        h = norm(x, w["post_attention_layernorm"])
        g, u = h @ w["mlp.gate_proj"].double().T, h @ w["mlp.up_proj"].double().T
        x = x + (g * torch.sigmoid(g) * u) @ w["mlp.down_proj"].double().T
    last = torch.tensor(new, device=DEV).cumsum(0) - 1
    h = norm(x[last], _normal(seed, "norm", HID, std=0.1, mean=1.0))
    head = _normal(seed, "head", VOCAB, HID, std=0.02)
    return {"logits": torch.cat([h @ c.double().T for c in head.split(16384)], 1)}


def _llama_work(case):
    sizes = _llama_sizes(case)
    rows, outs = sum(n for _, n in sizes), len(sizes)
    per_layer = HID * (HQ + 2 * HKV) * HD + HQ * HD * HID + 3 * HID * FF
    pairs = sum(n * a + n * (n + 1) // 2 for a, n in sizes)
    kv = sum(a + n for a, n in sizes) * 2 * HKV * HD * (1 if case["fp8_kv"] else 2)
    return {"bytes": 2 * (LAYERS * per_layer + HID * VOCAB) + LAYERS * kv + 4 * outs * VOCAB,
            "flops": 2 * (rows * LAYERS * per_layer + outs * HID * VOCAB) + LAYERS * pairs * 4 * HQ * HD}


# ------------------------------------------------------------------ mixture of experts
def _moe_weights(case, seed):
    E, _, H, I, _, gated = MOE[case["model"]]
    up = 2 * I if gated else I
    if not case["fp8"]:
        return _normal(seed, "w13", E, up, H, std=0.02), _normal(seed, "w2", E, H, I, std=0.02)
    out = []
    for tag, n, k in (("w13", up, H), ("w2", H, I)):
        q = torch.empty(E, n, k, dtype=torch.float8_e4m3fn, device=DEV)
        for a in range(0, E, 32):
            q[a:a + 32] = _normal(seed, tag + str(a), min(32, E - a), n, k, std=100.0).clamp_(-448, 448).to(q.dtype)
        scale = torch.empty(E, n // 128, k // 128, device=DEV).uniform_(1.6e-4, 2.5e-4, generator=_gen(seed, tag + "s"))
        out.append(Fp8Experts(q, scale))
    return out


def _moe_inputs(case, seed):
    """Normed rows, router logits (some experts are liked more than others) and the choice's bias."""
    E, _, H, _, router, _ = MOE[case["model"]]
    x = _normal(seed, "x", case["tokens"], H)
    logits = _normal(seed, "logits", case["tokens"], E, std=1.5, dtype=torch.float32) + _normal(seed, "liked", E, std=0.4, dtype=torch.float32)
    bias = None if router == "softmax" else _normal(seed, "bias", E, std=0.05, dtype=torch.float32)
    return x, logits, bias


def _moe_prepare(case, seed):
    w13, w2 = _moe_weights(case, seed)
    x, logits, bias = _moe_inputs(case, seed)
    return {"kind": "moe", "moe": MOE[case["model"]], "w13": w13, "w2": w2, "x": x, "logits": logits, "bias": bias}


def _moe_run(s):
    _, k, _, _, router, gated = s["moe"]
    if router == "softmax":
        w, ids = ops.moe_route(s["logits"], k)
    elif router == "sigmoid":
        w, ids = ops.moe_route(s["logits"], k, True, "sigmoid", bias=s["bias"], n_group=1, topk_group=1, group_mode=2)
    else:
        w, ids = ops.moe_route(s["logits"], k, True, "sigmoid", bias=s["bias"], n_group=8, topk_group=4, group_mode=2)
    out = ops.fused_moe(s["x"], w, ids, s["w13"], s["w2"], 0 if gated else 4, 1.0 if router == "softmax" else 2.5, gated=gated)
    return {"out": out, "weights": w, "ids": ids}


def _moe_exact(case, seed):
    E, k, H, I, router, gated = MOE[case["model"]]
    x, logits, bias = _moe_inputs(case, seed)
    logits = logits.double()
    if router == "softmax":
        score = choice = logits.softmax(-1)
    else:
        score = logits.sigmoid()
        choice = score + bias.double()
        if router == "groups":
            by = choice.view(len(x), 8, E // 8)
            keep = torch.zeros(len(x), 8, dtype=torch.bool, device=DEV)
            keep.scatter_(1, by.topk(2, -1).values.sum(-1).topk(4, -1).indices, True)
            choice = torch.where(keep[:, :, None], by, 0.0).view(len(x), E)
    ids = choice.topk(k, -1).indices
    w = score.gather(1, ids)
    w = w / w.sum(-1, keepdim=True)
    w13, w2 = _moe_weights(case, seed)

    def weight(t, e):
        if not case["fp8"]:
            return t[e].double()
        return t.q[e].double() * t.scale[e].double().repeat_interleave(128, 0).repeat_interleave(128, 1)

    out = torch.zeros(len(x), H, dtype=torch.float64, device=DEV)
    for e in range(E):
        row, slot = (ids == e).nonzero(as_tuple=True)
        if len(row):
            h = x[row].double() @ weight(w13, e).T
            h = h[:, :I] * h[:, :I].sigmoid() * h[:, I:] if gated else h.clamp(min=0).square()
            out.index_add_(0, row, h @ weight(w2, e).T * w[row, slot, None])
    return {"out": out * (1.0 if router == "softmax" else 2.5), "weights": w, "ids": None}


def _moe_work(case):
    E, k, H, I, _, gated = MOE[case["model"]]
    n, mats = case["tokens"] * k, 3 if gated else 2
    hit = E * (1 - (1 - k / E) ** case["tokens"])   # experts that some row chooses
    return {"bytes": hit * mats * H * I * (1 if case["fp8"] else 2) + case["tokens"] * (4 * H + 4 * E), "flops": 2.0 * n * mats * H * I}


# ------------------------------------------------------------------ multi-head latent attention
def _mla_sizes(case):
    """[(context, query rows)] of every sequence; the rows are its newest tokens."""
    if case["rows"] == 1:
        return [(n, 1) for n in _lens(case, "c", case["seqs"], case["ctx"])]
    past = case["ctx"] - case["rows"]
    return [(past + n, n) for n in _lens(case, "r", case["seqs"], case["rows"], 2)]


def _mla_inputs(case, seed):
    sizes = _mla_sizes(case)
    lat = _normal(seed, "lat", sum(c for c, _ in sizes), 576)
    q = _normal(seed, "q", sum(n for _, n in sizes), case["heads"], 576)
    return sizes, lat, q


MLA_SCALE = 192 ** -0.5


def _mla_prepare(case, seed):
    sizes, lat, q = _mla_inputs(case, seed)
    need = [-(-c // PAGE) for c, _ in sizes]
    pages = torch.randperm(sum(need), generator=torch.Generator().manual_seed(int(seed))) + 1
    cache = torch.zeros(sum(need) + 1, PAGE, 576, dtype=torch.bfloat16, device=DEV)
    table = torch.zeros(len(sizes), max(need), dtype=torch.int32)
    slots, p = [], 0
    for s, (c, _) in enumerate(sizes):
        own = pages[p:p + need[s]]
        p += need[s]
        table[s, :need[s]] = own.int()
        at = torch.arange(c)
        slots.append(own[at // PAGE] * PAGE + at % PAGE)
    cache.view(-1, 576)[torch.cat(slots).to(DEV)] = lat
    return {"kind": "mla", "q": q, "cache": cache, "table": table.to(DEV), "row": _i32([s for s, (_, n) in enumerate(sizes) for _ in range(n)]),
            "lens": _i32([c - n + 1 + j for c, n in sizes for j in range(n)]), "ws": ops.MLAWorkspace(DEV)}


def _mla_run(s):
    return {"out": ops.mla_attn(s["q"], s["cache"], s["table"], s["row"], s["lens"], MLA_SCALE, s["ws"])}


def _mla_exact(case, seed):
    sizes, lat, q = _mla_inputs(case, seed)
    out, a, b = [], 0, 0
    for c, n in sizes:
        kv = lat[a:a + c].double()
        for r in range(0, n, 256):
            m = min(256, n - r)
            sc = q[b + r:b + r + m].double() @ kv.T * MLA_SCALE
            seen = torch.arange(c, device=DEV)[None] <= torch.arange(c - n + r, c - n + r + m, device=DEV)[:, None]
            out.append(sc.masked_fill_(~seen[:, None], -math.inf).softmax(-1) @ kv[:, :512])
        a, b = a + c, b + n
    return {"out": torch.cat(out)}


def _mla_work(case):
    sizes = _mla_sizes(case)
    pairs = sum(n * (c - n) + n * (n + 1) // 2 for c, n in sizes)
    rows = sum(n for _, n in sizes)
    return {"bytes": 2 * (sum(c for c, _ in sizes) * 576 + rows * case["heads"] * (576 + 512)), "flops": 2 * pairs * case["heads"] * (576 + 512)}


# ------------------------------------------------------------------ recurrent layers
def _rec_sizes(case):
    """Rows of every sequence, and whether it starts here (a prompt) or goes on (a decode row)."""
    fresh = case["tokens"] > case["seqs"]
    return (_parts(case, "t", case["seqs"], case["tokens"]) if fresh else [1] * case["seqs"]), fresh


def _gdn_dims(case):
    hk, hv = 16 // case["shards"], 32 // case["shards"]
    return hk, hv, hk * 128, hv * 128


def _mamba_dims(case):
    return 128 // case["shards"], 8 // case["shards"]   # heads of 64, groups of 128 states


def _rec_values(case, seed):
    """The layer's in-projection rows, states, and constants (decays from nearly none to within a row)."""
    T, S, shards, gdn = case["tokens"], case["seqs"], case["shards"], case["kind"] == "gdn"
    if gdn:
        hk, hv, kd, vd = _gdn_dims(case)
        conv, width, heads, state = 2 * kd + vd, 2 * kd + 2 * vd + 2 * hv, hv, (hv, 128, 128)
        a = torch.log(torch.logspace(-1.7, 1.2, hv, device=DEV))
        dt_bias = torch.ones(hv, device=DEV)
    else:
        heads, groups = _mamba_dims(case)
        vd = heads * 64
        conv, width, state = vd + 2 * groups * 128, 2 * vd + 2 * groups * 128 + heads, (heads, 64, 128)
        a = -torch.logspace(0, 1.2, heads, device=DEV)
        dt_bias = torch.empty(heads, device=DEV).uniform_(-6.0, -2.0, generator=_gen(seed, "dt"))
    v = {"p": _normal(seed, "p", T, width), "conv_w": _normal(seed, "cw", conv, 4, std=0.3), "a": a, "dt_bias": dt_bias,
         "norm": _normal(seed, "norm", 128 if gdn else vd, std=0.1, mean=1.0), "conv_state": _normal(seed, "cs", S + 1, conv, 3),
         "state": _normal(seed, "st", S + 1, *state, std=0.1, dtype=torch.float32)}
    if not gdn:
        v["conv_b"] = _normal(seed, "cb", conv, std=0.1)
        v["d"] = _normal(seed, "d", heads, std=0.2, mean=1.0, dtype=torch.float32)
    return v


def _rec_prepare(case, seed):
    s = _rec_values(case, seed)
    rows, fresh = _rec_sizes(case)
    s["cu"] = _i32([sum(rows[:i]) for i in range(len(rows) + 1)])
    s["slot"] = _i32(list(range(len(rows))))
    s["reset"] = _i32([int(fresh)] * len(rows))
    s["kind"], s["dims"] = case["kind"], _gdn_dims(case) if case["kind"] == "gdn" else _mamba_dims(case)
    return s


def _gdn_run(s):
    hk, hv, kd, vd = s["dims"]
    p, cd, seqs = s["p"], 2 * kd + vd, (s["cu"], s["slot"], s["reset"])
    c = ops.ssm_conv1d(p[:, :cd], s["conv_w"], None, s["conv_state"], *seqs)
    o = ops.gdn_scan(c[:, :kd], c[:, kd:2 * kd], c[:, 2 * kd:], p[:, cd + vd + hv:], p[:, cd + vd:cd + vd + hv], s["a"], s["dt_bias"],
                     s["state"], *seqs, hv, hk)
    o = ops.gated_rmsnorm(o, p[:, cd:cd + vd], s["norm"], 128, 1e-6, norm_first=True)
    return {"out": o, "conv_state": s["conv_state"], "state": s["state"]}


def _mamba_run(s):
    heads, groups = s["dims"]
    vd, gn, seqs = heads * 64, groups * 128, (s["cu"], s["slot"], s["reset"])
    p, cd = s["p"], vd + 2 * gn
    c = ops.ssm_conv1d(p[:, vd:vd + cd], s["conv_w"], s["conv_b"], s["conv_state"], *seqs)
    y = ops.ssm_scan(c[:, :vd], p[:, vd + cd:], c[:, vd:vd + gn], c[:, vd + gn:], s["a"], s["d"], s["dt_bias"], 0.001, s["state"], *seqs,
                     heads, 64, 128, groups)
    y = ops.gated_rmsnorm(y, p[:, :vd], s["norm"], vd // groups, 1e-5)
    return {"out": y, "conv_state": s["conv_state"], "state": s["state"]}


def _rec_exact(case, seed):
    """Row by row over all sequences at once (padded to the longest)."""
    v = {k: t.double() for k, t in _rec_values(case, seed).items()}
    rows, fresh = _rec_sizes(case)
    S, L, T, gdn = len(rows), max(rows), case["tokens"], case["kind"] == "gdn"
    n = torch.tensor(rows, device=DEV)
    start = n.cumsum(0) - n
    at = (start[:, None] + torch.arange(L, device=DEV)).clamp(max=T - 1)
    live = torch.arange(L, device=DEV) < n[:, None]
    p = v["p"][at]
    if gdn:
        hk, hv, kd, vd = _gdn_dims(case)
        cd = 2 * kd + vd
        x, z = p[..., :cd], p[..., cd:cd + vd]
    else:
        heads, groups = _mamba_dims(case)
        vd, gn = heads * 64, groups * 128
        cd = vd + 2 * gn
        x, z = p[..., vd:vd + cd], p[..., :vd]
    before = torch.zeros_like(v["conv_state"][:S]) if fresh else v["conv_state"][:S]
    x = torch.cat([before.transpose(1, 2), x], 1)
    c = sum(x[:, j:j + L] * v["conv_w"][:, j] for j in range(4)) + (0 if gdn else v["conv_b"])
    c = c * c.sigmoid()
    tail = (n[:, None] + torch.arange(3, device=DEV))[:, :, None].expand(-1, -1, cd)
    conv_state, state = v["conv_state"].clone(), v["state"].clone()
    conv_state[:S] = x.gather(1, tail).transpose(1, 2)
    st = torch.zeros_like(state[:S]) if fresh else state[:S].clone()
    out = torch.zeros(S, L, vd, dtype=torch.float64, device=DEV)
    if gdn:
        q, k = (c[..., a:a + kd].view(S, L, hk, 128) for a in (0, kd))
        q, k = (t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt() for t in (q, k))
        q, k = (t.repeat_interleave(hv // hk, 2) for t in (q / math.sqrt(128), k))
        val = c[..., 2 * kd:].view(S, L, hv, 128)
        beta = p[..., cd + vd:cd + vd + hv].sigmoid()
        g = (-v["a"].exp() * torch.nn.functional.softplus(p[..., cd + vd + hv:] + v["dt_bias"])).exp()
        for t in range(L):
            on = live[:, t, None, None, None]
            s1 = st * g[:, t, :, None, None]
            u = (val[:, t] - (s1 @ k[:, t, :, :, None])[..., 0]) * beta[:, t, :, None]
            s1 = s1 + u[..., :, None] * k[:, t, :, None, :]
            out[:, t] = (s1 @ q[:, t, :, :, None]).reshape(S, vd)
            st = torch.where(on, s1, st)
        y = out.view(S, L, hv, 128)
        y = (y / (y.square().mean(-1, keepdim=True) + 1e-6).sqrt() * v["norm"]).view(S, L, vd) * z * z.sigmoid()
    else:
        xs = c[..., :vd].view(S, L, heads, 64)
        b, cc = (c[..., a:a + gn].view(S, L, groups, 128).repeat_interleave(heads // groups, 2) for a in (vd, vd + gn))
        dt = torch.nn.functional.softplus(p[..., vd + cd:] + v["dt_bias"]).clamp(min=0.001)
        da = (dt * v["a"]).exp()
        for t in range(L):
            on = live[:, t, None, None, None]
            s1 = st * da[:, t, :, None, None] + (dt[:, t, :, None] * xs[:, t])[..., :, None] * b[:, t, :, None, :]
            out[:, t] = ((s1 @ cc[:, t, :, :, None])[..., 0] + v["d"][:, None] * xs[:, t]).reshape(S, vd)
            st = torch.where(on, s1, st)
        y = (out * z * z.sigmoid()).view(S, L, groups, -1)
        y = (y / (y.square().mean(-1, keepdim=True) + 1e-5).sqrt()).view(S, L, vd) * v["norm"]
    state[:S] = st
    return {"out": y[live], "conv_state": conv_state, "state": state}


def _rec_work(case):
    T, S = case["tokens"], case["seqs"]
    _, fresh = _rec_sizes(case)
    if case["kind"] == "gdn":
        hk, hv, kd, vd = _gdn_dims(case)
        conv, width, cells, steps = 2 * kd + vd, 2 * kd + 2 * vd + 2 * hv, hv * 128 * 128, 7
    else:
        heads, groups = _mamba_dims(case)
        vd = heads * 64
        conv, width, cells, steps = vd + 2 * groups * 128, 2 * vd + 2 * groups * 128 + heads, heads * 64 * 128, 5
    return {"bytes": 2 * T * (width + vd) + (1 if fresh else 2) * S * (4 * cells + 6 * conv), "flops": T * (cells * steps + 8 * conv)}


# ------------------------------------------------------------------ the interface
def prepare(case, seed):
    return {"llama": _llama_prepare, "moe": _moe_prepare, "mla": _mla_prepare, "gdn": _rec_prepare, "mamba": _rec_prepare}[case["kind"]](case, seed)


@torch.no_grad()
def run(state):
    return {"llama": _llama_run, "moe": _moe_run, "mla": _mla_run, "gdn": _gdn_run, "mamba": _mamba_run}[state["kind"]](state)


@torch.no_grad()
def exact(case, seed):
    return {"llama": _llama_exact, "moe": _moe_exact, "mla": _mla_exact, "gdn": _rec_exact, "mamba": _rec_exact}[case["kind"]](case, seed)


def work(case):
    return {"llama": _llama_work, "moe": _moe_work, "mla": _mla_work, "gdn": _rec_work, "mamba": _rec_work}[case["kind"]](case)


def tolerance(case):
    """About four times the distance of the path from ``exact`` (0.0018 attention, 0.0039 bf16 experts, 0.0042
    recurrent layers: the bf16 stores).  A step of 32 bf16 layers is 0.02 off, and two orders of its sums as far
    from each other; fp8 experts round their activations to 8 bits, and a bf16 sum in another order moves some of them."""
    return {"rel": {"llama": 0.025, "moe": 0.02 if case.get("fp8") else 0.015, "mla": 0.007}.get(case["kind"], 0.015)}
