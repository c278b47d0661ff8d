"""The work a user of this package has it do, as timed cases.

Seven kinds of call, each through the package's public entry points, on a Llama-3-8B-shaped
FP8 KV cache (8 KV heads, 32 query heads, head_dim 128, pages of 16 tokens) unless a case
says otherwise:

* ``decode``   one query token per sequence attends to its FP8 pages;
* ``prefill``  blocks of new tokens attend to the FP8 pages (ring attention on one GPU);
* ``append``   new tokens are quantised and stored into pages (a prompt with dynamic
               scales, a decode step with the prompt's scales);
* ``gather``   pages are dequantised into contiguous bf16 K and V;
* ``heads``    a contiguous cache tensor is quantised per (layer, K/V, head) and back;
* ``int8``     the per-tensor int8 storage functions, there and back;
* ``belady``   the Belady tiering plan of a ring-attention schedule.
"""
from __future__ import annotations

import math
import random

import torch

from zenyx_amd import kv
from zenyx_amd.streaming.precision import dequantize_for_bf16_compute, quantize_to_fp8_storage
from zenyx_amd.train.belayd_kv_cache_tiering import RingAttentionAccessSequence
from zenyx_amd.train.fp8_kv_quantization import FP8KVQuantizer

_EXACT_MOST = 400_000_000  # values of an output that exact() computes in 64 bits


def listed():
    return [
        # One chat: the next token of a single sequence, one layer's attention.
        {"name": "decode_one", "kind": "decode", "seqs": 1, "lo": 2048, "hi": 2048, "q_heads": 32, "kv_heads": 8,
         "dim": 128, "page": 16},
        # A serving batch: 16 sequences of 1k-8k tokens, one layer's attention.
        {"name": "decode_batch", "kind": "decode", "seqs": 16, "lo": 1024, "hi": 8192, "q_heads": 32, "kv_heads": 8,
         "dim": 128, "page": 16},
        # A full long-context batch: 64 sequences at 32k, one layer's attention.
        {"name": "decode_long", "kind": "decode", "seqs": 64, "lo": 32768, "hi": 32768, "q_heads": 32,
         "kv_heads": 8, "dim": 128, "page": 16},
        # Several prompts at once: 4 x 8,192 tokens, causal, as a ring of 8.
        {"name": "prefill_full", "kind": "prefill", "seqs": 4, "q_lo": 8192, "q_hi": 8192, "old_lo": 0, "old_hi": 0,
         "ring": 8, "causal": True, "precision": "f16", "one_launch": True, "q_heads": 32, "kv_heads": 8, "page": 16},
        # Chunked prefill of a running server: two sequences' next chunks on top of what is cached.
        {"name": "prefill_chunk", "kind": "prefill", "seqs": 2, "q_lo": 300, "q_hi": 700, "old_lo": 4000,
         "old_hi": 12000, "ring": 1, "causal": True, "precision": "f16", "one_launch": True, "q_heads": 32,
         "kv_heads": 8, "page": 16},
        # A decode step's new tokens of all 32 layers, with the prompt's scales.
        {"name": "append_step", "kind": "append", "layers": 32, "seqs": 16, "lo": 1, "hi": 1, "old": 500,
         "static": True, "kv_heads": 8, "dim": 128, "page": 16},
        # 16 prompts of 1k-8k tokens, all 32 layers in one call.
        {"name": "append_prompt", "kind": "append", "layers": 32, "seqs": 16, "lo": 1024, "hi": 8192, "old": 0,
         "static": False, "kv_heads": 8, "dim": 128, "page": 16},
        # One layer of 4 x 32k tokens, as a cache streamed layer by layer appends it.
        {"name": "append_layer", "kind": "append", "layers": 1, "seqs": 4, "lo": 32768, "hi": 32768, "old": 0,
         "static": False, "kv_heads": 8, "dim": 128, "page": 16},
        # Decode through another attention: 64 x 32k tokens of one layer as bf16.
        {"name": "gather_long", "kind": "gather", "seqs": 64, "lo": 32768, "hi": 32768, "kv_heads": 8, "dim": 128,
         "page": 16},
        # A small model's whole cache (12 layers, 12 heads, 4,096 tokens of 64) to FP8 and back.
        {"name": "heads_roundtrip", "kind": "heads", "layers": 12, "batch": 1, "heads": 12, "tokens": 4096, "dim": 64},
        # One 4,096 x 4,096 bf16 tensor to int8 storage and back.
        {"name": "int8_storage", "kind": "int8", "n": 4096 * 4096, "dtype": "bfloat16"},
        # The tiering plan of 1M tokens x 80 layers in pages of 64 tokens, ring of 8, 64 GB of HBM.
        {"name": "belady_plan", "kind": "belady", "layers": 80, "ring": 8, "context": 1048576, "page": 64,
         "budget": 64e9},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "append", "append", "gather", "heads", "int8",
                       "belady"])
    page = rng.choice([16, 16, 32, 64])
    kv_heads, dim = rng.choice([(8, 128), (8, 128), (8, 128), (4, 128), (16, 128), (2, 128), (12, 64), (8, 64)])
    lens = random.Random(rng.randrange(1 << 30))  # of the case's sequence lengths
    if kind == "decode":
        seqs = _log(rng, 1, 64)
        hi = _log(rng, 100, 32768)
        return {"kind": kind, "seqs": seqs, "lo": max(1, hi // rng.choice([1, 2, 8])), "hi": hi,
                "q_heads": kv_heads * rng.choice([1, 4, 4, 8]), "kv_heads": kv_heads, "dim": dim, "page": page,
                "lens": lens.randrange(1 << 30)}
    if kind == "prefill":
        kv_heads = rng.choice([2, 4, 8, 8])
        seqs = rng.randint(1, 4)
        q_hi = _log(rng, 17, 8192)
        old = _log(rng, 1, 16384) if q_hi <= 2048 else 0
        return {"kind": kind, "seqs": seqs, "q_lo": max(1, q_hi // rng.choice([1, 2, 4])), "q_hi": q_hi,
                "old_lo": old // rng.choice([1, 2, 4]), "old_hi": old, "ring": rng.choice([1, 2, 4, 8]),
                "causal": rng.random() < 0.85, "precision": rng.choice(["f16", "f16", "f16", "bf16", "exact"]),
                "one_launch": rng.random() < 0.75, "q_heads": kv_heads * rng.choice([1, 2, 4, 4]),
                "kv_heads": kv_heads, "page": page, "lens": lens.randrange(1 << 30)}
    if kind == "append":
        static = rng.random() < 0.4
        seqs = _log(rng, 1, 64 if static else 16)
        layers = rng.choice([1, 1, 4, 12, 32])
        hi = _log(rng, 1, 16) if static else min(_log(rng, 50, 65536), 2_000_000 // (seqs * layers))
        return {"kind": kind, "layers": layers, "seqs": seqs, "lo": max(1, hi // rng.choice([1, 2, 4])), "hi": hi,
                "old": rng.randrange(500) if static else 0, "static": static, "kv_heads": kv_heads, "dim": dim,
                "page": page, "lens": lens.randrange(1 << 30)}
    if kind == "gather":
        seqs = _log(rng, 1, 64)
        hi = _log(rng, 100, 32768)
        return {"kind": kind, "seqs": seqs, "lo": max(1, hi // rng.choice([1, 2, 8])), "hi": hi,
                "kv_heads": kv_heads, "dim": dim, "page": rng.choice([page, 24]), "lens": lens.randrange(1 << 30)}
    if kind == "heads":
        layers, batch = rng.choice([1, 4, 12, 32]), rng.randint(1, 4)
        tokens = min(_log(rng, 65, 32768), 500_000_000 // (2 * layers * batch * kv_heads * dim))
        return {"kind": kind, "layers": layers, "batch": batch, "heads": kv_heads, "tokens": tokens, "dim": dim}
    if kind == "int8":
        return {"kind": kind, "n": _log(rng, 1000, 200_000_000),
                "dtype": rng.choice(["bfloat16", "bfloat16", "float16", "float32"])}
    layers, ring = _log(rng, 2, 80), rng.choice([2, 4, 8])
    shard = _log(rng, 64, 2048)
    pages = layers * ring * shard
    return {"kind": kind, "layers": layers, "ring": ring, "context": ring * shard * 64, "page": 64,
            "budget": float(int(pages * rng.uniform(0.2, 0.9)) * 64 * 8 * 128 * 2)}


# ---------------------------------------------------------------- sizes that a case gives

def _lengths(c, lo="lo", hi="hi", salt=0):
    r = random.Random(c.get("lens", 1) * 8 + salt)
    return [r.randint(c[lo], c[hi]) for _ in range(c["seqs"])]


def _prefill_sizes(c):
    new = _lengths(c, "q_lo", "q_hi")
    old = _lengths(c, "old_lo", "old_hi", 1)
    return new, old


def _pairs(c):
    """(query, key) pairs that count."""
    new, old = _prefill_sizes(c)
    return sum(n * o + (n * (n + 1) // 2 if c["causal"] else n * n) for n, o in zip(new, old))


def work(c):
    k = c["kind"]
    if k == "decode":
        tok = sum(_lengths(c))
        return {"bytes": 2 * tok * c["kv_heads"] * c["dim"] + 4 * c["seqs"] * c["q_heads"] * c["dim"],
                "flops": 4 * tok * c["q_heads"] * c["dim"]}
    if k == "prefill":
        new, old = _prefill_sizes(c)
        return {"bytes": 2 * (sum(new) + sum(old)) * c["kv_heads"] * 128 + 4 * sum(new) * c["q_heads"] * 128,
                "flops": 4 * 128 * c["q_heads"] * _pairs(c)}
    if k == "append":
        return {"bytes": 3 * c["layers"] * sum(_lengths(c)) * 2 * c["kv_heads"] * c["dim"], "flops": 0}
    if k == "gather":
        n = _lengths(c)
        return {"bytes": (sum(n) + 2 * c["seqs"] * max(n)) * 2 * c["kv_heads"] * c["dim"], "flops": 0}
    if k == "heads":
        return {"bytes": 5 * 2 * c["layers"] * c["batch"] * c["heads"] * c["tokens"] * c["dim"], "flops": 0}
    if k == "int8":
        return {"bytes": c["n"] * (_dtype(c).itemsize + 1 + 2), "flops": 0}
    return {"bytes": 5 * _trace_len(c), "flops": 0}


def _dtype(c):
    return getattr(torch, c["dtype"])


def _trace_len(c):
    shard = max(1, math.ceil(math.ceil(c["context"] / c["ring"]) / c["page"]))
    return 2 * c["layers"] * c["ring"] * c["ring"] * shard


def tolerance(c):
    """Attention is computed in 32 bits (the softmax weights of a prefill as its precision
    says) and rounded once to bf16; everything else is whole numbers, or 32-bit and bf16
    values that are each rounded once."""
    if c["kind"] in ("decode", "prefill"):
        return {"rel": 8e-3, "max": 5e-2}
    return "exact"


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(shape, g, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _ints(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def _tables(lens, page, g, spare):
    """Block tables over pages in random order, and the number of pages in the pool."""
    need = [-(-n // page) for n in lens]
    n_pages = sum(need) + spare
    order = torch.randperm(n_pages, generator=g, device="cuda").to(torch.int32)
    bt = torch.zeros((len(lens), max(max(need), 1)), dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = order[at:at + n]
        at += n
    return bt, n_pages


def _pool(n_pages, c, dim, g):
    """One layer's pages holding N(0, 1) keys and values as e4m3 codes, and its scales."""
    amax = 4.5 + torch.rand((2, c["kv_heads"]), generator=g, device="cuda")
    pool = torch.empty((n_pages, 2, c["kv_heads"], c["page"], dim), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 28) // pool[0].numel())
    for p in range(0, n_pages, step):
        x = _normal(pool[p:p + step].shape, g)
        pool[p:p + step] = (x * (448.0 / 5.0)).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    return pool, (amax / 448.0).contiguous()


def prepare(c, seed):
    g, k = _gen(seed), c["kind"]
    if k in ("decode", "gather"):
        lens = _lengths(c)
        bt, n_pages = _tables(lens, c["page"], g, 64)
        pool, scales = _pool(n_pages, c, c["dim"], g)
        s = {"case": c, "bt": bt, "pool": pool, "scales": scales, "lens": _ints(lens), "most": max(lens)}
        if k == "decode":
            s["q"] = _normal((c["seqs"], c["q_heads"], c["dim"]), g)
        return s
    if k == "prefill":
        new, old = _prefill_sizes(c)
        lens = [a + b for a, b in zip(new, old)]
        bt, n_pages = _tables(lens, c["page"], g, 64)
        pool, scales = _pool(n_pages, c, 128, g)
        cu = [0]
        for n in new:
            cu.append(cu[-1] + n)
        return {"case": c, "bt": bt, "pool": pool, "scales": scales, "lens": _ints(lens), "cu": _ints(cu),
                "pos0": _ints(old), "most": max(new), "q": _normal((cu[-1], c["q_heads"], 128), g)}
    if k == "append":
        new = _lengths(c)
        r = random.Random(c.get("lens", 1) * 8 + 3)
        old = [r.randint(c["old"] // 2, c["old"]) for _ in new]
        bt, n_pages = _tables([a + b for a, b in zip(new, old)], c["page"], g, 8)
        x = _normal((c["layers"], sum(new), 2, c["kv_heads"], c["dim"]), g)
        # some heads of a trained model run far larger than the others
        big = 1 + 49 * (torch.rand((c["layers"], 1, 2, c["kv_heads"], 1), generator=g, device="cuda") < 0.05)
        for layer in range(c["layers"]):
            x[layer] *= big[layer].to(torch.bfloat16)
        cu = [0]
        for n in new:
            cu.append(cu[-1] + n)
        pool = torch.zeros((c["layers"], n_pages, 2, c["kv_heads"], c["page"], c["dim"]), dtype=torch.uint8,
                           device="cuda")
        scales = (6.0 / 448.0) * big.reshape(c["layers"], 2, c["kv_heads"]).float().contiguous()
        return {"case": c, "x": x, "cu": _ints(cu), "start": _ints(old), "bt": bt, "pool": pool, "scales": scales}
    if k == "heads":
        x = _normal((c["layers"], 2, c["batch"], c["heads"], c["tokens"], c["dim"]), g)
        return {"case": c, "x": x, "quantizer": FP8KVQuantizer()}
    if k == "int8":
        return {"case": c, "x": _normal((c["n"],), g, _dtype(c))}
    # The schedule itself has no random part; the pages' numbers start where the allocator stood.
    shard = max(1, math.ceil(math.ceil(c["context"] / c["ring"]) / c["page"]))
    order = RingAttentionAccessSequence(c["layers"], c["ring"], shard)
    trace = (order.trace("cuda") + seed * 7919 % order.n_pages) % order.n_pages
    page_bytes = c["page"] * 8 * 128 * 2
    return {"case": c, "trace": trace, "n_pages": order.n_pages,
            "capacity": max(1, min(order.n_pages, int(c["budget"] // page_bytes)))}


# ---------------------------------------------------------------- one pass

def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "decode":
        return kv.paged_attention_decode(s["q"], s["pool"], s["scales"], s["bt"], s["lens"])
    if k == "prefill":
        return kv.ring_attention_fp8(s["q"], s["cu"], s["pos0"], s["pool"], s["scales"], s["bt"], s["lens"],
                                     c["ring"], causal=c["causal"], precision=c["precision"],
                                     single_launch=c["one_launch"], max_q_per_seq=s["most"])
    if k == "append":
        if c["static"]:
            scales = kv.kv_quant_append(s["x"], s["cu"], s["bt"], s["pool"], scales=s["scales"],
                                        start_pos=s["start"], static_scales=True)
        else:
            scales = kv.kv_quant_append(s["x"], s["cu"], s["bt"], s["pool"], start_pos=s["start"])
        return s["pool"], scales
    if k == "gather":
        return kv.kv_gather_dequant(s["pool"], s["scales"], s["bt"], s["lens"], s["most"])
    if k == "heads":
        codes, scales = s["quantizer"].quantize(s["x"])
        return codes, scales, s["quantizer"].dequantize(codes, scales)
    if k == "int8":
        q, scale = quantize_to_fp8_storage(s["x"])
        return q, scale, dequantize_for_bf16_compute(q, scale)
    sim = kv.BeladyTraceSim(s["trace"], s["n_pages"], s["capacity"], record_misses=True)
    sim.run()
    n = sim.n_evicted
    return sim.state, sim.evict_pos[:n], sim.evict_page[:n], sim.miss_flags


# ---------------------------------------------------------------- in 64 bits

def _values(codes):
    return codes.view(torch.float8_e4m3fn).to(torch.float32).double()


def _cached(s, b, n):
    """K and V of sequence b's first n positions, [heads, n, dim] in 64 bits."""
    page = s["case"]["page"]
    rows = s["pool"][s["bt"][b, :-(-n // page)].long()]  # [pages, 2, heads, page, dim]
    rows = rows.permute(1, 2, 0, 3, 4).flatten(2, 3)[:, :, :n]
    v = _values(rows.contiguous()) * s["scales"].double()[:, :, None, None]
    return v[0], v[1]


def exact(c, seed):
    k = c["kind"]
    if k == "belady":
        return None
    s = prepare(c, seed)
    if k == "decode":
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        for b, n in enumerate(_lengths(c)):
            kk, vv = _cached(s, b, n)
            q = s["q"][b].double().view(c["kv_heads"], -1, c["dim"])
            w = torch.softmax(torch.matmul(q, kk.transpose(1, 2).contiguous()) * c["dim"] ** -0.5, dim=-1)
            out[b] = torch.matmul(w, vv).reshape(-1, c["dim"])
        return out
    if k == "prefill":
        new, old = _prefill_sizes(c)
        if _pairs(c) * c["q_heads"] > 8e9:
            return None
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        at, per = 0, c["q_heads"] // c["kv_heads"]
        for b, (n, o) in enumerate(zip(new, old)):
            kk, vv = _cached(s, b, n + o)
            for h in range(c["q_heads"]):
                for r in range(0, n, 4096):
                    q = s["q"][at + r:at + min(n, r + 4096), h].double()
                    w = torch.matmul(q, kk[h // per].t().contiguous()) * 128 ** -0.5
                    if c["causal"]:
                        pos = o + r + torch.arange(q.shape[0], device="cuda")
                        w.masked_fill_(torch.arange(n + o, device="cuda")[None, :] > pos[:, None], -math.inf)
                    out[at + r:at + r + q.shape[0], h] = torch.matmul(torch.softmax(w, dim=-1), vv[h // per])
            at += n
        return out
    if k == "append":
        if c["static"]:
            return None, s["scales"].double()
        amax = torch.stack([x.abs().amax(dim=(0, 3)).double() for x in s["x"]])
        return None, amax.clamp_min(1e-8) / 448.0
    if k == "gather":
        n = _lengths(c)
        if c["seqs"] * max(n) * c["kv_heads"] * c["dim"] > _EXACT_MOST:
            return None
        ko = torch.zeros((c["seqs"], c["kv_heads"], max(n), c["dim"]), dtype=torch.float64, device="cuda")
        vo = torch.zeros_like(ko)
        for b, m in enumerate(n):
            ko[b, :, :m], vo[b, :, :m] = _cached(s, b, m)
        return ko, vo
    if k == "heads":
        amax = s["x"].abs().amax(dim=(2, 4, 5)).double()
        return None, amax.clamp_min(1e-8) / 448.0, None
    amax = s["x"].abs().amax().double()
    return None, amax.clamp_min(1e-8) / 127.0, None
