"""The work a serving engine has this library do, as cases that can be timed and compared.

Kinds of case:

  step      one engine step of the Llama-3-8B-shaped model (`aici_amd.llama`): the batch's index arrays go to the
            device, every layer runs over its own paged KV cache, and the AICI allow-mask and the arg-max end the step.
            `rows` sequences decode one token each; `chunks` more bring `new_lo`..`new_hi` tokens of a prompt.
  decode    one layer's paged decode attention (`kernels.paged_attention_v1`).
  prefill   one layer's prompt pass: the new keys and values go into the cache (`kernels.reshape_and_cache`), then causal
            attention over the rows of k / v, or over the cache through block tables.
  mixed     one layer's attention of a continuous-batching step (`attn.varlen_attn`): prompt chunks over what is cached
            already, beside decode rows.
  sample    the AICI mask with temperature and top-p over a batch's logits (`kernels.bias_sample`).
  fork      copy-on-write copies of cache blocks in every layer (`paged.CacheEngine.copy`).

The lengths of a case's sequences come from the case alone (`spread` seeds them); the seed of `prepare` makes the values,
the order of the blocks in the pool and the weights.
"""
import math

import numpy as np
import torch

from aici_amd import attn, kernels, llama, paged
from aici_amd import workloads as W

BLOCK = 16
LLAMA_HEADS, PHI2_HEADS, NARROW_HEADS = (32, 8, 128), (32, 32, 80), (16, 2, 64)
MHA_HEADS = (32, 32, 128)
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
VOCAB = 128256


def _heads(shape):
    return {"query_heads": shape[0], "kv_heads": shape[1], "head_size": shape[2]}


def listed():
    return [
        # A single chat: one sequence of the full 32-layer model, as an interactive user waits for it.
        {"name": "step_1", "kind": "step", "dtype": "bf16", "layers": 32, "rows": 1, "ctx_lo": 700, "ctx_hi": 700,
         "chunks": 0, "new_lo": 0, "new_hi": 0, "prior_hi": 0, "spread": 1},
        # A small server: sixteen sequences of the full 32-layer model.
        {"name": "step_16", "kind": "step", "dtype": "bf16", "layers": 32, "rows": 16, "ctx_lo": 256, "ctx_hi": 2048,
         "chunks": 0, "new_lo": 0, "new_hi": 0, "prior_hi": 0, "spread": 2},
        # A full server: the benchmark's 128 sequences over contexts U[1k,16k] (four of its layers: a state of all 32
        # takes 160 GB).
        {"name": "step_128", "kind": "step", "dtype": "bf16", "layers": 4, "rows": 128, "ctx_lo": 1024, "ctx_hi": 16384,
         "chunks": 0, "new_lo": 0, "new_hi": 0, "prior_hi": 0, "spread": 5},
        # Continuous batching: prompts arrive (some with a cached prefix) while other sequences generate.
        {"name": "step_chunked", "kind": "step", "dtype": "bf16", "layers": 8, "rows": 24, "ctx_lo": 128,
         "ctx_hi": 4096, "chunks": 4, "new_lo": 17, "new_hi": 512, "prior_hi": 1024, "spread": 3},
        # Few short contexts, multi-head attention at head size 80: where launches and latency count.
        {"name": "decode_short", "kind": "decode", "dtype": "fp16", **_heads(PHI2_HEADS), "rows": 8, "ctx_lo": 16,
         "ctx_hi": 512, "spread": 8},
        # The benchmark's decode configuration.
        {"name": "decode_64", "kind": "decode", "dtype": "bf16", **_heads(LLAMA_HEADS), "rows": 64, "ctx_lo": 512,
         "ctx_hi": 4096, "spread": 2},
        # Four short prompts, multi-head attention in fp16, with their cache write (the parity configuration's sizes).
        {"name": "prefill_short", "kind": "prefill", "dtype": "fp16", **_heads(MHA_HEADS), "seqs": 4, "len_lo": 128,
         "len_hi": 512, "paged": False, "spread": 0},
        # A batch of prompts of very different lengths, narrow heads, read through block tables.
        {"name": "prefill_ragged", "kind": "prefill", "dtype": "fp16", **_heads(NARROW_HEADS), "seqs": 32, "len_lo": 1,
         "len_hi": 2048, "paged": True, "spread": 4},
        # The benchmark's prefill configuration: long prompts.
        {"name": "prefill_long", "kind": "prefill", "dtype": "bf16", **_heads(LLAMA_HEADS), "seqs": 8, "len_lo": 4096,
         "len_hi": 4096, "paged": False, "spread": 3},
        # The benchmark's mixed step: four 512-token chunks over cached prefixes, 120 decode rows, by the default route.
        {"name": "mixed", "kind": "mixed", "dtype": "fp16", **_heads(PHI2_HEADS), "rows": 120, "ctx_lo": 1024,
         "ctx_hi": 8192, "chunks": 4, "new_lo": 512, "new_hi": 512, "prior_hi": 3072, "paged": False, "spread": 4},
        # The sampling end of a step: every row with its own allow-mask, temperature and nucleus.
        {"name": "sample_128", "kind": "sample", "dtype": "bf16", "rows": 128, "vocab": VOCAB, "allowed": 0.05,
         "top_p": 0.9, "temperature": 0.8},
        # A batch of sequences forks: one shared block each to be copied, in all 32 layers.
        {"name": "fork_16", "kind": "fork", "dtype": "bf16", **_heads(LLAMA_HEADS), "layers": 32, "pairs": 16},
    ]


# --------------------------------------------------------------------------- drawn cases

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _span(rng, lo, hi):
    """Two ends of a range of lengths within [lo, hi]."""
    top = _log(rng, lo, hi)
    return max(lo, int(top * rng.choice([0.05, 0.25, 0.5, 1.0]))), top


def _fits(case, nbytes, flops):
    """Whether a drawn case asks for no more than these."""
    w = work(case)
    return w["bytes"] <= nbytes and w["flops"] <= flops


def draw(rng):
    kind = rng.choice(["step", "step", "step", "decode", "decode", "prefill", "prefill", "mixed", "sample", "fork"])
    c = {"kind": kind, "dtype": rng.choice(["bf16", "fp16"])}
    spread = rng.randrange(1 << 20)
    if kind == "step":
        c.update(layers=rng.choice([1, 2, 4, 8, 16, 32]), rows=_log(rng, 1, 128), chunks=0, new_lo=0, new_hi=0, prior_hi=0)
        c["ctx_lo"], c["ctx_hi"] = _span(rng, 16, 16384)
        if rng.random() < 0.35:
            c["chunks"] = rng.randint(1, 6)
            c["new_lo"], c["new_hi"] = _span(rng, 2, 700)
            c["prior_hi"] = rng.choice([0, 0, 500, 2000])
            c["layers"] = min(c["layers"], 8)
        while not _fits(dict(c, spread=spread), 20e9, 3e12):
            if c["layers"] > 1:
                c["layers"] //= 2
            else:
                c["rows"] = max(1, c["rows"] // 2)
    elif kind == "decode":
        c.update(_heads(rng.choice([LLAMA_HEADS, LLAMA_HEADS, PHI2_HEADS, NARROW_HEADS, MHA_HEADS])), rows=_log(rng, 1, 128))
        c["ctx_lo"], c["ctx_hi"] = _span(rng, 16, 16384)
        while not _fits(dict(c, spread=spread), 6e9, 1e12):
            c["rows"] = max(1, c["rows"] // 2)
    elif kind == "prefill":
        c.update(_heads(rng.choice([LLAMA_HEADS, LLAMA_HEADS, PHI2_HEADS, NARROW_HEADS, MHA_HEADS])), seqs=_log(rng, 1, 64),
                 paged=rng.random() < 0.5)
        c["len_lo"], c["len_hi"] = _span(rng, 2, 8192)
        while not _fits(dict(c, spread=spread), 1e9, 1.1e12):
            c["seqs"] = max(1, c["seqs"] // 2)
    elif kind == "mixed":
        c.update(_heads(rng.choice([LLAMA_HEADS, PHI2_HEADS])), rows=_log(rng, 1, 120), chunks=rng.randint(1, 6),
                 prior_hi=rng.choice([0, 500, 3000]), paged=rng.random() < 0.5)
        c["ctx_lo"], c["ctx_hi"] = _span(rng, 16, 8192)
        c["new_lo"], c["new_hi"] = _span(rng, 2, 700)
        while not _fits(dict(c, spread=spread), 6e9, 1e12):
            c["rows"] = max(1, c["rows"] // 2)
    elif kind == "sample":
        c.update(rows=_log(rng, 1, 256), vocab=rng.choice([VOCAB, 51200, 32000, rng.randint(1000, VOCAB)]),
                 allowed=rng.choice([0.0005, 0.05, 1.0]), top_p=rng.choice([1.0, 0.95, 0.9, 0.5]),
                 temperature=round(rng.uniform(0.3, 1.5), 2))
    else:
        c.update(_heads(rng.choice([LLAMA_HEADS, PHI2_HEADS, MHA_HEADS])), layers=rng.choice([8, 24, 32]),
                 pairs=_log(rng, 1, 128))
    c["spread"] = spread
    return c


# --------------------------------------------------------------------------- sizes

def _entries(case):
    """(length, tokens computed already) of every sequence: the decode rows last, as the engine orders them."""
    rng = np.random.default_rng(case["spread"])
    out = []
    for i in range(case.get("chunks", 0)):
        new = int(rng.integers(case["new_lo"], case["new_hi"] + 1))
        prior = 0 if i == 0 else int(case["prior_hi"] * i // max(1, case["chunks"] - 1))
        out.append((prior + new, prior))
    for n in rng.integers(case["ctx_lo"], case["ctx_hi"] + 1, size=case["rows"]).tolist():
        out.append((n, n - 1))
    return out


def _lens(case):
    rng = np.random.default_rng(case["spread"])
    lens = rng.integers(case["len_lo"], case["len_hi"] + 1, size=case["seqs"]).tolist()
    return sorted(lens, key=lambda n: n == 1)  # one-token prompts last, where the engine's batch puts them


def _shape(case):
    if case["kind"] == "step":
        return LLAMA_HEADS
    return case["query_heads"], case["kv_heads"], case["head_size"]


def _kv_bytes(case):
    _, hkv, d = _shape(case)
    return sum(n for n, _ in _entries(case)) * 2 * hkv * d * 2 * case.get("layers", 1)


def _attention_flops(entries, hq, d):
    """Two products over the unmasked (query, key) pairs."""
    return 4 * d * hq * sum((n - c) * c + (n - c) * (n - c + 1) // 2 for n, c in entries)


def work(case):
    kind = case["kind"]
    if kind == "step":
        cfg = llama.LlamaConfig.llama3_8b()
        hidden, ffn, vocab, layers = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, case["layers"]
        entries = _entries(case)
        tokens, rows = sum(n - c for n, c in entries), len(entries)
        weights = layers * (hidden * hidden * 2 + hidden * 2048 + 3 * hidden * ffn)
        moved = 2 * (weights + vocab * hidden) + _kv_bytes(case) + 2 * rows * vocab
        flops = 2 * weights * tokens + 2 * vocab * hidden * rows + layers * _attention_flops(entries, 32, 128)
        return {"bytes": moved, "flops": flops}
    if kind == "sample":
        return {"bytes": case["rows"] * (2 * case["vocab"] + case["vocab"] // 8), "flops": 0}
    hq, hkv, d = _shape(case)
    if kind == "fork":
        return {"bytes": 2 * case["pairs"] * case["layers"] * 2 * hkv * d * BLOCK * 2, "flops": 0}
    if kind == "prefill":
        entries = [(n, 0) for n in _lens(case)]
        tokens = sum(n for n, _ in entries)
        # q in, output out, k and v in, and into the cache
        return {"bytes": 2 * tokens * d * (2 * hq + 4 * hkv), "flops": _attention_flops(entries, hq, d)}
    entries = _entries(case)
    tokens = sum(n - c for n, c in entries)
    scatter = 0 if kind == "decode" else 4 * tokens * hkv * d * 2
    return {"bytes": _kv_bytes(case) + 2 * tokens * hq * d * 2 + scatter, "flops": _attention_flops(entries, hq, d)}


def tolerance(case):
    kind = case["kind"]
    if kind == "fork":
        return "exact"
    if kind == "sample":
        # a draw within rounding of an edge of the cumulative sum may fall on its other side
        return {"rel": 0.0, "differ": 0.01}
    if kind == "step":
        # Every product summed in another order, carried through the layers in 16 bits.  Measured against products
        # in fp32 rounded once, bf16: 2.3e-3 / 3.4e-3 / 8.5e-3 at 4 / 8 / 32 layers (largest 1.0e-2 / 1.5e-2 / 4.1e-2).
        rel = (5e-3 if case["dtype"] == "bf16" else 1e-3) * math.sqrt(case["layers"])
        return {"rel": rel, "max": 6 * rel}
    # Measured between the launch strategies and kernels: bf16 2.5e-3 (largest 4.3e-2), fp16 2.0e-4 (3.6e-3).
    return {"rel": 1e-2, "max": 0.17} if case["dtype"] == "bf16" else {"rel": 8e-4, "max": 0.015}


# --------------------------------------------------------------------------- inputs

def _batch(entries, rng, vocab):
    """The engine's block allocator (its free list in a random order, as after a while of serving) and the step's batch."""
    need = sum((n + BLOCK - 1) // BLOCK for n, _ in entries)
    pool = need + 64
    alloc = paged.BlockAllocator(BLOCK, pool)
    for sid in range(pool):  # one block each, given back in a random order
        alloc.alloc_seq(1_000_000 + sid, BLOCK)
    for sid in rng.permutation(pool).tolist():
        alloc.delete(1_000_000 + sid)
    builder = paged.BatchInfoBuilder(BLOCK, 1 << 20, 1)
    for sid, (n, computed) in enumerate(entries, start=1):
        alloc.alloc_seq(sid, n)
        builder.sched_out(alloc, sid, rng.integers(0, vocab, size=n).astype(np.int32), computed)
    return pool, builder.finish()


def _packed_masks(rows, vocab, share, g, dev):
    """Packed allow-bits [rows, 4 * ceil(vocab / 32)], bit k of byte i for token 8i + k."""
    width = (vocab + 31) // 32 * 32
    allowed = torch.rand((rows, width), generator=g, device=dev) < share
    allowed[:, 0] = True
    allowed[:, vocab:] = False
    bits = (1 << torch.arange(8, device=dev, dtype=torch.int32)).to(torch.uint8)
    return (allowed.view(rows, width // 8, 8).to(torch.uint8) * bits).sum(-1, dtype=torch.uint8)


def _prepare_step(case, rng, g, dev):
    cfg = llama.LlamaConfig.llama3_8b()
    cfg.num_hidden_layers = case["layers"]
    cfg.dtype = DTYPES[case["dtype"]]
    entries = _entries(case)
    pool, batch = _batch(entries, rng, cfg.vocab_size)
    # A residual stream as a trained model's: its layers add to it, they do not replace it.
    weights = llama.random_weights(cfg, int(rng.integers(1 << 30)), device=dev, std=0.006)
    weights["model.embed_tokens"].mul_(1 / 0.006)
    model = llama.Llama(cfg, weights, dev)
    del weights
    hkv, d = cfg.num_key_value_heads, cfg.head_dim
    keys = torch.empty((case["layers"], pool, hkv, d // 8, BLOCK, 8), dtype=cfg.dtype, device=dev).normal_(generator=g)
    values = torch.empty((case["layers"], pool, hkv, d, BLOCK), dtype=cfg.dtype, device=dev).normal_(generator=g)
    return {"batch": batch, "model": model, "keys": keys, "values": values, "device": dev,
            "caches": [(keys[i], values[i]) for i in range(case["layers"])],
            "masks": _packed_masks(len(entries), cfg.vocab_size, 0.05, g, dev)}


def _normal(shape, dtype, g, dev):
    return torch.randn(shape, generator=g, device=dev, dtype=dtype)


def _cache(pool, hkv, d, dtype, g, dev):
    kc, vc = paged.alloc_gpu_cache_layer(pool, hkv, d, BLOCK, dtype, dev)
    return kc.normal_(generator=g), vc.normal_(generator=g)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)
    rng = np.random.default_rng(seed)
    if kind == "step":
        state = _prepare_step(case, rng, g, dev)
    elif kind == "sample":
        rows, vocab = case["rows"], case["vocab"]
        # a few tokens stand out of the rest, as a trained model's do
        logits = _normal((rows, vocab), torch.float32, g, dev) * 2.0
        logits.scatter_add_(1, torch.randint(0, vocab, (rows, 32), generator=g, device=dev),
                            torch.rand((rows, 32), generator=g, device=dev) * 8.0)
        state = {"logits": logits.to(dtype), "masks": _packed_masks(rows, vocab, case["allowed"], g, dev),
                 "temperature": torch.full((rows,), case["temperature"], device=dev),
                 "top_p": torch.full((rows,), case["top_p"], device=dev),
                 "uniforms": torch.rand((rows,), generator=g, device=dev)}
    elif kind == "fork":
        _, hkv, d = _shape(case)
        pairs = case["pairs"]
        engine = paged.CacheEngine(case["layers"], hkv, d, BLOCK, dtype, 2 * pairs + 16, 0, dev)
        for kc, vc in engine.gpu_cache:
            kc.normal_(generator=g)
            vc.normal_(generator=g)
        blocks = rng.permutation(2 * pairs + 16).tolist()
        state = {"engine": engine, "copies": {blocks[i]: [blocks[pairs + i]] for i in range(pairs)}}
    else:
        hq, hkv, d = _shape(case)
        entries = [(n, 0) for n in _lens(case)] if kind == "prefill" else _entries(case)
        pool, batch = _batch(entries, rng, 1000)
        tokens = batch.tokens.numel()
        kc, vc = _cache(pool, hkv, d, dtype, g, dev)
        state = {"batch": batch.to(dev), "kc": kc, "vc": vc, "q": _normal((tokens, hq, d), dtype, g, dev),
                 "scale": 1.0 / math.sqrt(d), "hkv": hkv, "paged": case.get("paged", False)}
        if kind == "decode":
            state["out"] = torch.empty_like(state["q"])
        else:
            state["k"], state["v"] = (_normal((tokens, hkv, d), dtype, g, dev) for _ in range(2))
            if kind == "prefill":
                state["offsets"] = W.offsets([n for n, _ in entries]).to(dev)
                state["longest"] = max(n for n, _ in entries)
                state["context_lens"] = torch.tensor([n for n, _ in entries], dtype=torch.int32, device=dev)
                tables = _tables(batch, entries)
                state["tables"] = tables.to(dev)
    state["kind"] = kind
    return state


def _tables(batch, entries):
    """Block tables of prompts that start empty, from the slots their tokens go to."""
    width = max((n + BLOCK - 1) // BLOCK for n, _ in entries)
    tables = torch.zeros((len(entries), width), dtype=torch.int32)
    at = 0
    for i, (n, _) in enumerate(entries):
        blocks = batch.slot_mapping[at:at + n:BLOCK] // BLOCK
        tables[i, :blocks.numel()] = blocks
        at += n
    return tables


# --------------------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "step":
        logits = state["model"].forward(state["batch"].to(state["device"]), state["caches"], paged_prefill=True, fused=True)
        # The token that wins is left out of what is returned: random weights leave near-ties that a sum taken in
        # another order decides the other way.  Its logit is compared instead.
        _, best = kernels.bias_argmax(logits, mask=state["masks"], return_logits=True)
        return {"logits": logits, "best": best, "keys": state["keys"], "values": state["values"]}
    if kind == "decode":
        b = state["batch"]
        kernels.paged_attention_v1(state["out"], state["q"], state["kc"], state["vc"], state["hkv"], state["scale"],
                                   b.paged_block_tables, b.paged_context_lens, BLOCK, b.paged_max_context_len)
        return state["out"]
    if kind == "prefill":
        kernels.reshape_and_cache(state["k"], state["v"], state["kc"], state["vc"], state["batch"].slot_mapping)
        if state["paged"]:
            out = kernels.flash_attn_varlen_paged(state["q"], state["kc"], state["vc"], state["tables"], state["offsets"],
                                                  state["context_lens"], state["longest"], state["longest"], state["scale"])
        else:
            out = kernels.flash_attn_varlen(state["q"], state["k"], state["v"], state["offsets"], state["offsets"],
                                            state["longest"], state["longest"], state["scale"], True)
        return {"out": out, "keys": state["kc"], "values": state["vc"]}
    if kind == "mixed":
        y = attn.varlen_attn(state["q"], state["k"], state["v"], state["batch"], state["kc"], state["vc"], state["scale"],
                             paged_prefill=state["paged"])
        return {"out": y, "keys": state["kc"], "values": state["vc"]}
    if kind == "sample":
        return kernels.bias_sample(state["logits"], state["temperature"], state["top_p"], state["uniforms"],
                                   mask=state["masks"])
    state["engine"].copy(state["copies"])
    return [t for pair in state["engine"].gpu_cache for t in pair]
