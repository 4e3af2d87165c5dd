"""What this framework's users have it do, as cases that can be timed and checked.

Five kinds of call, each through the public entry points:

* ``decode``  -- paged decode attention of one step (``paged_decode_attention``, or the
  ``PagedDecodePlan`` that a decode loop keeps);
* ``prompt``  -- causal attention over one prompt (``flash_prefill_attention``) and, with
  ``write``, the K/V write of the same layer from its slot mapping (``KVCache.write_kv_slots``);
* ``packed``  -- causal attention over several prompts in one launch (``flash_prefill_varlen``);
* ``pass``    -- a prompt, or a chunk of one after a cached prefix, through a model
  (``Llama.prefill_table``); one or two layers stand for the blocks of one;
* ``step``    -- one batched decode step of a model through its captured graph (``DecodeGraph``).

Integers (context lengths, block tables, prompt lengths) come from numpy, values from a seeded
generator on the device: N(0, 1) activations, as RMSNorm and the projections leave them, and
model weights of N(0, 0.02).
"""

import math

import numpy as np
import torch

from tinyvllm_amd.attention import (PagedDecodePlan, flash_prefill_attention, flash_prefill_varlen,
                                    paged_decode_attention)
from tinyvllm_amd.kv_cache import KVCache
from tinyvllm_amd.llama import DecodeGraph, Llama, LlamaConfig

DEVICE = "cuda"
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}

# (query heads, KV heads, head size): TinyLlama, Llama-3-8B and its 4-way shard
HEADS = {"tinyllama": (32, 4, 64), "llama3_8b": (32, 8, 128), "llama3_8b_shard": (8, 2, 128)}

# (dim, query heads, KV heads, hidden): TinyLlama, LlamaConfig's defaults with grouped heads, a small one
SHAPES = {"tinyllama": (2048, 32, 4, 5632), "wide": (4096, 32, 8, 16384), "small": (1024, 16, 4, 2816)}
VOCAB = 32000


def listed():
    return [
        # The smallest call: an interactive engine of four short conversations in the reference's
        # default type, attention of one layer through the drop-in function.
        {"name": "decode_f32_few", "kind": "decode", "dtype": "float32", "heads": "tinyllama", "block": 16,
         "batch": 4, "ctx_min": 17, "ctx_max": 250, "plan": False},
        # A full serving batch of mixed context lengths, as a decode loop launches it.
        {"name": "decode_f16_batch", "kind": "decode", "dtype": "float16", "heads": "llama3_8b", "block": 16,
         "batch": 256, "ctx_min": 512, "ctx_max": 4096, "plan": True},
        # A few sequences of very long context: the split-context path.
        {"name": "decode_bf16_long", "kind": "decode", "dtype": "bfloat16", "heads": "llama3_8b", "block": 16,
         "batch": 16, "ctx_min": 32768, "ctx_max": 32768, "plan": True},
        # One layer's attention and K/V write for an ordinary prompt.
        {"name": "prompt_f16", "kind": "prompt", "dtype": "float16", "heads": "tinyllama", "block": 16,
         "length": 1000, "write": True},
        # A long document.
        {"name": "prompt_bf16_long", "kind": "prompt", "dtype": "bfloat16", "heads": "llama3_8b", "block": 16,
         "length": 8192, "write": False},
        # The reference's default type.
        {"name": "prompt_f32", "kind": "prompt", "dtype": "float32", "heads": "tinyllama", "block": 16,
         "length": 512, "write": True},
        # A batch of new requests of unequal length, attended together.
        {"name": "packed_f16", "kind": "packed", "dtype": "float16", "heads": "tinyllama", "count": 12,
         "len_min": 30, "len_max": 1500},
        # A layer and the head of a long prompt's second chunk, over the cached first one.
        {"name": "chunk_bf16_block", "kind": "pass", "dtype": "bfloat16", "shape": "wide", "layers": 1, "block": 16,
         "length": 2048, "start": 2048, "logits": "last"},
        # Two layers of a short prompt in the reference's default type, with the logits of every
        # token as the reference's prefill returns them.
        {"name": "pass_f32_block", "kind": "pass", "dtype": "float32", "shape": "tinyllama", "layers": 2, "block": 16,
         "length": 300, "start": 0, "logits": "all"},
        # A whole model's prompt: the time to the first token.
        {"name": "pass_f16_model", "kind": "pass", "dtype": "float16", "shape": "tinyllama", "layers": 22,
         "block": 16, "length": 1000, "start": 0, "logits": "last"},
        # Two layers and the head of an interactive engine's step in the reference's default type.
        {"name": "step_f32_few", "kind": "step", "dtype": "float32", "shape": "tinyllama", "layers": 2, "block": 16,
         "batch": 4, "ctx_min": 17, "ctx_max": 250},
        # A whole model's decode step at a serving batch: what every generated token costs.
        {"name": "step_f16_model", "kind": "step", "dtype": "float16", "shape": "tinyllama", "layers": 22,
         "block": 16, "batch": 64, "ctx_min": 1000, "ctx_max": 1152},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "packed", "pass", "pass", "step", "step"])
    dtype = rng.choice(["float32", "float16", "bfloat16"])
    block = rng.choice([16, 16, 32])
    if kind == "decode":
        heads = rng.choice(sorted(HEADS))
        batch = _log_int(rng, 1, 256)
        row = 2 * HEADS[heads][1] * HEADS[heads][2] * DTYPES[dtype].itemsize
        most = max(64, min(32768, (2 << 30) // (row * batch)))
        ctx = _log_int(rng, 64, most)
        return {"kind": kind, "dtype": dtype, "heads": heads, "block": block, "batch": batch,
                "ctx_min": max(1, int(ctx * rng.uniform(0.1, 1.0))), "ctx_max": ctx, "plan": rng.random() < 0.5}
    if kind == "prompt":
        most = 1500 if dtype == "float32" else 8192
        return {"kind": kind, "dtype": dtype, "heads": rng.choice(sorted(HEADS)), "block": block,
                "length": _log_int(rng, 16, most), "write": rng.random() < 0.5}
    if kind == "packed":
        longest = _log_int(rng, 64, 2048)
        return {"kind": kind, "dtype": rng.choice(["float16", "bfloat16"]), "heads": rng.choice(sorted(HEADS)),
                "count": _log_int(rng, 2, 24), "len_min": max(1, longest // rng.choice([2, 8, 32])),
                "len_max": longest}
    shape = rng.choice(sorted(SHAPES))
    if kind == "pass":
        length = _log_int(rng, 8, 512 if dtype == "float32" else 2048)
        start = rng.choice([0, 0, _log_int(rng, 16, 2048)])
        return {"kind": kind, "dtype": dtype, "shape": shape, "layers": rng.choice([1, 2]), "block": block,
                "length": length, "start": start, "logits": rng.choice(["last", "all"])}
    ctx = _log_int(rng, 32, 2048)
    return {"kind": kind, "dtype": dtype, "shape": shape, "layers": rng.choice([1, 2]), "block": block,
            "batch": _log_int(rng, 1, 64), "ctx_min": max(1, int(ctx * rng.uniform(0.1, 1.0))), "ctx_max": ctx}


# ---- inputs -------------------------------------------------------------------------

def _ints(seed, stream):
    return np.random.Generator(np.random.PCG64([seed, stream]))


def _floats(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return gen


def _normal(gen, shape, dtype, std=1.0):
    x = torch.randn(shape, generator=gen, dtype=dtype, device=DEVICE)
    return x if std == 1.0 else x.mul_(std)


def _contexts(case, seed):
    """Context lengths: the case's own, dealt to the sequences by the seed."""
    ctx = _ints(0, 1).integers(case["ctx_min"], case["ctx_max"] + 1, case["batch"]).astype(np.int32)
    return _ints(seed, 1).permutation(ctx)


def _tables(lens, block, seed):
    """Block tables of sequences of `lens` positions over a shuffled pool with a tenth to spare."""
    need = -(-np.asarray(lens, dtype=np.int64) // block)
    pool = int(need.sum() * 1.1) + 1
    perm = _ints(seed, 2).permutation(pool).astype(np.int32)
    table = np.zeros((len(need), int(need.max())), np.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    return table, pool


def _lengths(case, seed):
    """Prompt lengths: the case's own, in the seed's order."""
    lens = _ints(0, 3).integers(case["len_min"], case["len_max"] + 1, case["count"])
    return [int(n) for n in _ints(seed, 3).permutation(lens)]


def _decode_inputs(case, seed):
    hq, hkv, d = HEADS[case["heads"]]
    dtype, block = DTYPES[case["dtype"]], case["block"]
    ctx = _contexts(case, seed)
    table, pool = _tables(ctx, block, seed)
    gen = _floats(seed)
    q = _normal(gen, (case["batch"], 1, hq, d), dtype)
    k = _normal(gen, (pool, block, hkv, d), dtype)
    v = _normal(gen, (pool, block, hkv, d), dtype)
    return q, k, v, torch.from_numpy(table).to(DEVICE), torch.from_numpy(ctx).to(DEVICE)


def _prompt_inputs(case, seed):
    hq, hkv, d = HEADS[case["heads"]]
    dtype, n = DTYPES[case["dtype"]], case["length"]
    gen = _floats(seed)
    return tuple(_normal(gen, (1, n, h, d), dtype) for h in (hq, hkv, hkv))


def _slots(table, block, start, count):
    pos = np.arange(start, start + count)
    return (table[pos // block].astype(np.int64) * block + pos % block).astype(np.int32)


def _packed_inputs(case, seed):
    hq, hkv, d = HEADS[case["heads"]]
    lens = _lengths(case, seed)
    gen = _floats(seed)
    return lens, tuple(_normal(gen, (sum(lens), h, d), DTYPES[case["dtype"]]) for h in (hq, hkv, hkv))


def _weights(case, seed):
    dim, hq, hkv, hidden = SHAPES[case["shape"]]
    d = dim // hq
    dtype = DTYPES[case["dtype"]]
    gen = _floats(seed + 7)
    w = {"tok_embeddings.weight": _normal(gen, (VOCAB, dim), dtype, 0.02),
         "output.weight": _normal(gen, (VOCAB, dim), dtype, 0.02),
         "norm.weight": 1 + _normal(gen, (dim,), torch.float32, 0.1)}
    for i in range(case["layers"]):
        for name, shape in (("attention.wq", (hq * d, dim)), ("attention.wk", (hkv * d, dim)),
                            ("attention.wv", (hkv * d, dim)), ("attention.wo", (dim, hq * d)),
                            ("feed_forward.w1", (hidden, dim)), ("feed_forward.w3", (hidden, dim)),
                            ("feed_forward.w2", (dim, hidden))):
            w[f"layers.{i}.{name}.weight"] = _normal(gen, shape, dtype, 0.02)
        for name in ("attention_norm", "ffn_norm"):
            w[f"layers.{i}.{name}.weight"] = 1 + _normal(gen, (dim,), torch.float32, 0.1)
    return w


def _model_inputs(case, seed):
    """Tokens, positions, tables and the cached K/V of the model kinds."""
    dim, hq, hkv, _ = SHAPES[case["shape"]]
    d = dim // hq
    dtype, block = DTYPES[case["dtype"]], case["block"]
    if case["kind"] == "pass":
        lens = np.asarray([case["start"] + case["length"]])
        tokens = _ints(seed, 4).integers(0, VOCAB, case["length"]).astype(np.int32)
    else:
        lens = _contexts(case, seed)            # the step's own position is the last one attended
        tokens = _ints(seed, 4).integers(0, VOCAB, case["batch"]).astype(np.int32)
    table, pool = _tables(lens, block, seed)
    gen = _floats(seed + 13)
    # keys and values of unit-RMS activations through N(0, 0.02) projections
    fill = case["kind"] == "step" or case["start"] > 0
    cached = [[_normal(gen, (pool, block, hkv, d), dtype, 0.02 * math.sqrt(dim)) if fill else
               torch.zeros((pool, block, hkv, d), dtype=dtype, device=DEVICE) for _ in range(case["layers"])]
              for _ in range(2)]
    return tokens, lens, table, pool, cached


def _model(case, seed):
    dim, hq, hkv, hidden = SHAPES[case["shape"]]
    config = LlamaConfig(dim=dim, n_layers=case["layers"], n_heads=hq, n_kv_heads=hkv, vocab_size=VOCAB,
                         hidden_dim=hidden, max_seq_len=4096, dtype=case["dtype"])
    tokens, lens, table, pool, cached = _model_inputs(case, seed)
    model = Llama(config, _weights(case, seed), device=DEVICE)
    cache = KVCache(case["layers"], pool, case["block"], hkv, dim // hq, case["dtype"], DEVICE)
    for mine, given in zip((cache.k_cache, cache.v_cache), cached):
        for t, x in zip(mine, given):
            t.copy_(x)
    return model, cache, tokens, lens, table


# ---- the passes ---------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        hq, hkv, d = HEADS[case["heads"]]
        args = (*_decode_inputs(case, seed), hq, hkv, d, case["block"])
        return {"kind": kind, "args": args, "plan": PagedDecodePlan(*args) if case["plan"] else None}
    if kind == "prompt":
        _, hkv, d = HEADS[case["heads"]]
        q, k, v = _prompt_inputs(case, seed)
        state = {"kind": kind, "q": q, "k": k, "v": v, "cache": None}
        if case["write"]:
            table, pool = _tables([case["length"]], case["block"], seed)
            state["cache"] = KVCache(1, pool, case["block"], hkv, d, case["dtype"], DEVICE)
            state["slots"] = torch.from_numpy(_slots(table[0], case["block"], 0, case["length"])).to(DEVICE)
        return state
    if kind == "packed":
        lens, (q, k, v) = _packed_inputs(case, seed)
        return {"kind": kind, "q": q, "k": k, "v": v, "lens": lens}
    model, cache, tokens, lens, table = _model(case, seed)
    state = {"kind": kind, "model": model, "cache": cache, "tokens": torch.from_numpy(tokens).to(DEVICE)}
    if kind == "pass":
        state.update(table=torch.from_numpy(table[0]).to(DEVICE), start=case["start"], logits=case["logits"])
        return state
    state.update(positions=torch.from_numpy(lens - 1).to(DEVICE), lens=torch.from_numpy(lens).to(DEVICE),
                 tables=torch.from_numpy(table).to(DEVICE),
                 graph=DecodeGraph(model, cache, case["batch"], table.shape[1]))
    state["graph"].capture()
    return state


def run(state):
    kind = state["kind"]
    if kind == "decode":
        return state["plan"].run() if state["plan"] else paged_decode_attention(*state["args"])
    if kind == "prompt":
        cache = state["cache"]
        if cache is None:
            return flash_prefill_attention(state["q"], state["k"], state["v"])
        cache.write_kv_slots(0, state["slots"], state["k"][0], state["v"][0])
        return [flash_prefill_attention(state["q"], state["k"], state["v"]), cache.k_cache[0], cache.v_cache[0]]
    if kind == "packed":
        return flash_prefill_varlen(state["q"], state["k"], state["v"], state["lens"])
    cache = state["cache"]
    if kind == "pass":
        logits = state["model"].prefill_table(state["tokens"], cache, state["table"], state["start"],
                                              logits=state["logits"], attend_prefix=state["start"] > 0)
        return {"logits": logits, "k": cache.k_cache, "v": cache.v_cache}
    graph = state["graph"]
    graph.set_inputs(state["tokens"], state["positions"], state["lens"], state["tables"])
    graph.step()
    return {"logits": graph.logits, "k": cache.k_cache, "v": cache.v_cache}


# ---- what a pass cannot do without --------------------------------------------------

def _pairs(length, start=0):
    """(query, key) pairs of `length` causal rows after `start` keys."""
    return length * start + length * (length + 1) // 2


def _mean_ctx(case):
    return (case["ctx_min"] + case["ctx_max"]) / 2


def work(case):
    es = DTYPES[case["dtype"]].itemsize
    kind = case["kind"]
    if kind in ("decode", "prompt", "packed"):
        hq, hkv, d = HEADS[case["heads"]]
        if kind == "decode":
            tokens = case["batch"] * _mean_ctx(case)
            return {"bytes": es * d * (2 * hkv * tokens + 2 * hq * case["batch"]) + 4 * tokens / case["block"],
                    "flops": 4 * hq * d * tokens}
        if kind == "prompt":
            n, write = case["length"], case["write"]
            return {"bytes": es * d * n * (2 * hq + 2 * hkv * (2 if write else 1)) + (4 * n if write else 0),
                    "flops": 4 * hq * d * _pairs(n)}
        lo, hi = case["len_min"], case["len_max"]
        n, square = (lo + hi) / 2, (lo * lo + lo * hi + hi * hi) / 3
        return {"bytes": es * d * case["count"] * n * (2 * hq + 2 * hkv),
                "flops": 4 * hq * d * case["count"] * (square + n) / 2}
    dim, hq, hkv, hidden = SHAPES[case["shape"]]
    d = dim // hq
    layer = dim * (2 * hq + 2 * hkv) * d + 3 * dim * hidden      # weights of one layer
    if kind == "pass":
        n, start = case["length"], case["start"]
        heads_rows = n if case["logits"] == "all" else 1
        pairs, cached = _pairs(n, start), start
        embedded, written = n, n
    else:
        n = heads_rows = embedded = written = case["batch"]
        pairs = cached = n * _mean_ctx(case)
    moved = es * (case["layers"] * layer + VOCAB * dim + embedded * dim +
                  case["layers"] * 2 * hkv * d * (cached + written)) + 4 * VOCAB * heads_rows
    return {"bytes": moved, "flops": 2 * n * case["layers"] * layer + case["layers"] * 4 * hq * d * pairs +
            2 * heads_rows * VOCAB * dim}


def tolerance(case):
    """About four times the error against 64 bits that was measured over listed and drawn cases:
    the rounding of one attention's output and weights, or of all of a model's layers."""
    dtype = case["dtype"]
    if case["kind"] in ("decode", "prompt", "packed"):
        return {"rel": {"float32": 2e-6, "float16": 1.5e-3, "bfloat16": 8e-3}[dtype]}
    return {"rel": {"float32": 2e-5, "float16": 6e-3, "bfloat16": 3e-2}[dtype]}


# ---- the same in 64 bits, plain torch ------------------------------------------------

def _attend(q, k, v, start=0, causal=True):
    """q [n, Hq, D] at positions start.., k / v [m, Hkv, D], all float64."""
    n, hq, d = q.shape
    group = hq // k.shape[1]
    out = torch.empty_like(q)
    for h in range(hq):
        s = q[:, h] @ k[:, h // group].T.contiguous() / math.sqrt(d)
        if causal:
            s.masked_fill_(torch.ones(s.shape, dtype=torch.bool, device=s.device).triu_(start + 1), -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // group].contiguous()
    return out


def _attend_one(q, k, v):
    """One query row [Hq, D] over k / v [m, Hkv, D], float64."""
    hq, d = q.shape
    hkv = k.shape[1]
    q = q.view(hkv, hq // hkv, d)
    s = torch.matmul(q, k.permute(1, 2, 0).contiguous()) / math.sqrt(d)
    return torch.matmul(torch.softmax(s, -1), v.transpose(0, 1).contiguous()).reshape(hq, d)


def _rows(cache, table, count):
    block = cache.shape[1]
    ids = torch.as_tensor(table[:-(-count // block)].astype(np.int64), device=cache.device)
    return cache[ids].reshape(-1, *cache.shape[2:])[:count].double()


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double()


def _rope(x, positions):
    """x [n, H, D]: pairs (2i, 2i + 1) turned by position * 10000^(-2i / D)."""
    d = x.shape[-1]
    freq = 10000.0 ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    angle = positions.double()[:, None, None] * freq
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()], -1).flatten(-2)


def _exact_model(case, seed):
    dim, hq, hkv, _ = SHAPES[case["shape"]]
    d, block = dim // hq, case["block"]
    tokens, lens, table, _, (k_cache, v_cache) = _model_inputs(case, seed)
    w = _weights(case, seed)
    if case["kind"] == "pass":
        positions = np.arange(case["start"], case["start"] + case["length"])
        slots = _slots(table[0], block, case["start"], case["length"])
    else:
        positions = lens - 1
        slots = table[np.arange(len(lens)), positions // block].astype(np.int64) * block + positions % block
    positions = torch.as_tensor(positions, device=DEVICE)
    slots = torch.as_tensor(slots.astype(np.int64), device=DEVICE)
    x = w["tok_embeddings.weight"][torch.as_tensor(tokens.astype(np.int64), device=DEVICE)].double()
    n = x.shape[0]
    written = {"k": [], "v": []}
    for i in range(case["layers"]):
        def mul(a, name):
            return a @ w[f"layers.{i}.{name}.weight"].double().T.contiguous()
        a = _norm(x, w[f"layers.{i}.attention_norm.weight"])
        q = _rope(mul(a, "attention.wq").view(n, hq, d), positions)
        k = _rope(mul(a, "attention.wk").view(n, hkv, d), positions)
        v = mul(a, "attention.wv").view(n, hkv, d)
        for name, cache, new in (("k", k_cache[i], k), ("v", v_cache[i], v)):
            cache = cache.double()
            cache.view(-1, hkv, d)[slots] = new
            written[name].append(cache)
        kc, vc = written["k"][-1], written["v"][-1]
        if case["kind"] == "pass":
            m = case["start"] + n
            o = _attend(q, _rows(kc, table[0], m), _rows(vc, table[0], m), case["start"])
        else:
            o = torch.stack([_attend_one(q[b], _rows(kc, table[b], int(lens[b])), _rows(vc, table[b], int(lens[b])))
                             for b in range(n)])
        x = x + mul(o.reshape(n, hq * d), "attention.wo")
        a = _norm(x, w[f"layers.{i}.ffn_norm.weight"])
        x = x + mul(torch.nn.functional.silu(mul(a, "feed_forward.w1")) * mul(a, "feed_forward.w3"),
                    "feed_forward.w2")
    x = _norm(x, w["norm.weight"])
    if case["kind"] == "pass" and case["logits"] == "last":
        x = x[-1:]
    logits = x @ w["output.weight"].double().T.contiguous()
    return {"logits": logits[None] if case["kind"] == "pass" else logits, **written}


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        q, k, v, table, ctx = _decode_inputs(case, seed)
        table, ctx = table.cpu().numpy(), ctx.cpu().numpy()
        return torch.stack([_attend_one(q[b, 0].double(), _rows(k, table[b], int(ctx[b])),
                                        _rows(v, table[b], int(ctx[b]))) for b in range(len(ctx))])[:, None]
    if kind == "prompt":
        q, k, v = _prompt_inputs(case, seed)
        out = _attend(q[0].double(), k[0].double(), v[0].double())[None]
        if not case["write"]:
            return out
        table, pool = _tables([case["length"]], case["block"], seed)
        slots = torch.as_tensor(_slots(table[0], case["block"], 0, case["length"]).astype(np.int64), device=DEVICE)
        caches = []
        for x in (k, v):
            c = torch.zeros((pool, case["block"], *x.shape[2:]), dtype=torch.float64, device=DEVICE)
            c.view(-1, *x.shape[2:])[slots] = x[0].double()
            caches.append(c)
        return [out, *caches]
    if kind == "packed":
        lens, (q, k, v) = _packed_inputs(case, seed)
        parts, at = [], 0
        for n in lens:
            parts.append(_attend(*(t[at:at + n].double() for t in (q, k, v))))
            at += n
        return torch.cat(parts)
    return _exact_model(case, seed)
