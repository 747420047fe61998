"""The framework's measured workloads: paged decode attention, cache writes, the elementwise steps
of a prefill layer and a whole decode step, each through its public entry points.

``listed()`` names twelve cases, ``draw(rng)`` gives further ones of the same ranges.  A case is a
dict of plain values; ``prepare(case, seed)`` makes its inputs on the GPU from the seed alone,
``run(state)`` is one pass, ``work(case)`` the bytes and operations a pass cannot do without,
``exact(case, seed)`` its results in 64 bits by plain torch, ``tolerance(case)`` how far another
correct implementation at the same precision may be off.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "int8-kvcache_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import int8kv  # noqa: E402
from int8kv import cache_ops, decode_loop  # noqa: E402
from int8kv import synthetic as syn  # noqa: E402

DEV = "cuda"
DTYPES = {"int8": torch.int8, "bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"int8": 1, "bf16": 2, "fp16": 2, "fp32": 4}

# Elements of the largest listed decode's K (or V) cache: drawn ones stay below.
MOST_CACHE_ELEMENTS = 64 * 16384 * 4 * 128


# ------------------------------------------------------------------------------------- cases
def _decode(name, batch, longest, hq, hkv, d, *, cache="int8", query="bf16", block=16,
            ragged=False, lens=0, quantize_q=False, append=False):
    return {"name": name, "kind": "decode", "batch": batch, "longest": longest, "hq": hq,
            "hkv": hkv, "d": d, "cache": cache, "query": query, "block": block, "ragged": ragged,
            "lens": lens, "quantize_q": quantize_q, "append": append}


def listed():
    return [
        # One short conversation, one layer's attention: nothing but latency and launches.
        _decode("int8_1x512", 1, 512, 28, 4, 128),
        # A small serving batch: one layer of a decode step as the serving glue calls it, the new
        # tokens' cache write and then the attention.
        _decode("int8_append_8x4096", 8, 4096, 28, 4, 128, append=True),
        # The benchmark's batch: contexts anywhere up to 32k tokens, the cache far larger than any
        # on-chip memory.
        _decode("int8_64x32k_ragged", 64, 32768, 28, 4, 128, ragged=True, lens=3),
        # The 16-bit cache the INT8 one is compared with, at a medium serving batch.
        _decode("bf16_32x8k", 32, 8192, 28, 4, 128, cache="bf16"),
        # 64-wide heads (Llama-3.2-1B's 32 / 8), an odd batch of ragged chats.
        _decode("int8_hd64_45x4k_ragged", 45, 4099, 32, 8, 64, ragged=True, lens=5),
        # 256-wide heads (Gemma-2-9B's 16 / 8), fp16 activations.
        _decode("int8_hd256_20x6k_ragged", 20, 6001, 16, 8, 256, query="fp16", ragged=True, lens=7),
        # One kv head per query head and a head size between the powers of two (Phi-3-mini's
        # 32 x 96), vLLM's larger block.
        _decode("int8_mha96_12x4k_ragged", 12, 4000, 32, 32, 96, block=32, ragged=True, lens=9),
        # Multi-query attention (Falcon-7B's 71 query heads on one kv head).
        _decode("int8_mqa71_40x4k", 40, 4096, 71, 1, 64),
        # A prefill's cache write: 8 prompts of 2048 tokens, some padding slots.
        {"name": "write_16k", "kind": "write", "tokens": 16384, "padding": 512, "hkv": 4, "d": 128,
         "source": "bf16", "block": 16, "dynamic": False},
        # A large prefill's cache write with a scale per token and head, an odd token count.
        {"name": "write_dynamic_100k", "kind": "write", "tokens": 100003, "padding": 0, "hkv": 8,
         "d": 128, "source": "fp16", "block": 16, "dynamic": True},
        # The library's own steps of one prefill layer over a chunk of prompts: two residual adds
        # with RMSNorm, rotary embedding, the cache write, SwiGLU.
        {"name": "prefill_layer_ops_6k", "kind": "prefill_ops", "tokens": 6007},
        # One decode step of the loop (graph replay), six of its 28 layers and the LM head, 32
        # sequences of 8k tokens.
        {"name": "decode_step_32x8k", "kind": "step", "batch": 32, "context": 8191, "layers": 6,
         "cache": "int8"},
    ]


SHAPES = [  # (query heads, kv heads, head_dim) of the tests and benchmarks
    (28, 4, 128), (28, 4, 128), (28, 4, 128), (32, 8, 128), (32, 8, 64), (14, 2, 64), (16, 8, 256),
    (8, 1, 256), (32, 32, 96), (32, 32, 80), (71, 1, 64)]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 6 + ["write"] * 2 + ["prefill_ops", "step"])
    if kind == "decode":
        hq, hkv, d = rng.choice(SHAPES)
        cache = rng.choice(["int8", "int8", "int8", "bf16", "fp16"])
        query = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        batch = _log_int(rng, 1, 160)
        most = MOST_CACHE_ELEMENTS // (batch * hkv * d * SIZE[cache])
        return {"kind": kind, "batch": batch, "longest": _log_int(rng, 16, min(32768, most)),
                "hq": hq, "hkv": hkv, "d": d, "cache": cache, "query": query,
                "block": rng.choice([16, 16, 32]), "ragged": rng.random() < 0.6,
                "lens": rng.randrange(1000), "quantize_q": cache == "int8" and rng.random() < 0.1,
                "append": cache == "int8" and rng.random() < 0.3}
    if kind == "write":
        dynamic = rng.random() < 0.4
        hkv, d = rng.choice([(4, 128), (8, 128), (8, 64), (8, 256)] + ([] if dynamic else [(2, 80)]))
        source = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        tokens = _log_int(rng, 1, 200_000_000 // (hkv * d * SIZE[source]))
        return {"kind": kind, "tokens": tokens, "padding": rng.randrange(0, 64), "hkv": hkv, "d": d,
                "source": source, "block": rng.choice([16, 32]), "dynamic": dynamic}
    if kind == "prefill_ops":
        return {"kind": kind, "tokens": _log_int(rng, 33, 6007)}
    cache = rng.choice(["int8", "int8", "bf16"])
    return {"kind": kind, "batch": _log_int(rng, 1, 32 // SIZE[cache]),
            "context": _log_int(rng, 64, 8191), "layers": rng.randrange(2, 7), "cache": cache}


# ------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _channels(hkv, d, g):
    """Per (kv head, channel) multiplier and offset of K: a few outlier channels, a mean offset."""
    mult = torch.ones(hkv, d, device=DEV)
    outliers = torch.rand(hkv, d, generator=g, device=DEV).topk(4, dim=1).indices
    mult.scatter_(1, outliers, 8.0)
    return mult, torch.randn(hkv, d, generator=g, device=DEV) * 0.5


def _sample_kv(n, mult, offset, g, dtype):
    hkv, d = mult.shape
    k = torch.randn(n, hkv, d, generator=g, device=DEV).mul_(mult).add_(offset)
    v = torch.randn(n, hkv, d, generator=g, device=DEV).mul_(0.5)
    return k.to(dtype), v.to(dtype)


def _static_scales(mult, offset, g):
    """absmax / 127 per kv head over a 4096-token sample, as the calibration does."""
    k, v = _sample_kv(4096, mult, offset, g, torch.float32)
    return tuple((t.abs().amax(dim=(0, 2)) / 127.0).clamp_min(1e-6) for t in (k, v))


def _quantised(x, scale):
    return (x.float() / scale[:, None]).round().clamp(-127, 127).to(torch.int8)


def _fill_caches(blocks, block, mult, offset, cache, ks, vs, g):
    """K and V caches [blocks, block, Hkv, D] holding sampled rows (INT8: quantised)."""
    hkv, d = mult.shape
    shape = (blocks, block, hkv, d)
    kc = torch.empty(shape, dtype=DTYPES[cache], device=DEV)
    vc = torch.empty_like(kc)
    step = max(1, (1 << 25) // (block * hkv * d))
    for b0 in range(0, blocks, step):
        n = min(step, blocks - b0)
        k, v = _sample_kv(n * block, mult, offset, g, torch.bfloat16)
        if cache == "int8":
            k, v = _quantised(k, ks), _quantised(v, vs)
        kc[b0:b0 + n].copy_(k.view(n, block, hkv, d))
        vc[b0:b0 + n].copy_(v.view(n, block, hkv, d))
    return kc, vc


def _lengths(case):
    if case["ragged"]:
        return [int(x) for x in syn.ragged_lengths(case["batch"], case["longest"], case["lens"])]
    return [case["longest"]] * case["batch"]


def _tables(lens, block, g):
    """[B, width] int32 tables over one shuffled pool shared by all sequences."""
    need = [-(-n // block) for n in lens]
    pool = torch.randperm(sum(need), generator=g, device=DEV).to(torch.int32)
    tables = torch.zeros(len(lens), max(need), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = pool[at:at + n]
        at += n
    return tables, sum(need)


def _decode_inputs(case, seed):
    g = _generator(seed)
    lens = _lengths(case)
    hq, hkv, d, block = case["hq"], case["hkv"], case["d"], case["block"]
    mult, offset = _channels(hkv, d, g)
    ks, vs = _static_scales(mult, offset, g)
    tables, blocks = _tables(lens, block, g)
    kc, vc = _fill_caches(blocks, block, mult, offset, case["cache"], ks, vs, g)
    q = torch.randn(len(lens), hq, d, generator=g, device=DEV).to(DTYPES[case["query"]])
    last = torch.tensor([n - 1 for n in lens], dtype=torch.int64, device=DEV)
    new_k, new_v = _sample_kv(len(lens), mult, offset, g, torch.bfloat16)
    slots = tables.gather(1, (last // block)[:, None])[:, 0].to(torch.int64) * block + last % block
    return {"kind": "decode", "q": q, "kc": kc, "vc": vc, "tables": tables,
            "lens": (last + 1).to(torch.int32), "ks": ks, "vs": vs, "new_k": new_k, "new_v": new_v,
            "slots": slots, "cache": case["cache"], "quantize_q": case["quantize_q"],
            "append": case["append"]}


def _write_inputs(case, seed):
    g = _generator(seed)
    n, hkv, d, block = case["tokens"], case["hkv"], case["d"], case["block"]
    mult, offset = _channels(hkv, d, g)
    ks, vs = _static_scales(mult, offset, g)
    rows = n + case["padding"]
    k, v = _sample_kv(rows, mult, offset, g, DTYPES[case["source"]])
    blocks = -(-n // block) + 2
    slots = torch.full((rows,), -1, dtype=torch.int64, device=DEV)
    valid = torch.randperm(rows, generator=g, device=DEV)[:n].sort().values
    # Whole blocks in shuffled order, as a paged allocator hands them out, each filled in order.
    pool = torch.randperm(blocks, generator=g, device=DEV)
    t = torch.arange(n, device=DEV)
    slots[valid] = pool[t // block] * block + t % block
    kc = torch.zeros(blocks, block, hkv, d, dtype=torch.int8, device=DEV)
    state = {"kind": "write", "k": k, "v": v, "kc": kc, "vc": torch.zeros_like(kc), "slots": slots,
             "ks": ks, "vs": vs, "dynamic": case["dynamic"]}
    if case["dynamic"]:
        state["ksc"] = torch.zeros(blocks, block, hkv, device=DEV)
        state["vsc"] = torch.zeros(blocks, block, hkv, device=DEV)
    return state


def _prefill_inputs(case, seed):
    g = _generator(seed)
    shape = decode_loop.QWEN25_7B
    n = case["tokens"]

    def normal(*size, std=1.0):
        return torch.empty(*size, dtype=torch.bfloat16, device=DEV).normal_(0.0, std, generator=g)

    blocks = -(-n // 16)
    pool = torch.randperm(blocks, generator=g, device=DEV)
    t = torch.arange(n, device=DEV)
    kc = torch.zeros(blocks, 16, shape.kv_heads, shape.head_dim, dtype=torch.int8, device=DEV)
    half = shape.head_dim // 2
    freq = shape.rope_theta ** (torch.arange(half, dtype=torch.float64, device=DEV) * -2.0 / shape.head_dim)
    ang = t.double()[:, None] * freq[None, :]
    ang = torch.cat([ang, ang], dim=1)
    return {"kind": "prefill_ops", "shape": shape, "x": normal(n, shape.hidden),
            "attn_out": normal(n, shape.hidden, std=0.5), "mlp_out": normal(n, shape.hidden, std=0.5),
            "w1": normal(shape.hidden, std=0.1) + 1, "w2": normal(shape.hidden, std=0.1) + 1,
            "h": torch.empty(n, shape.hidden, dtype=torch.bfloat16, device=DEV),
            "h2": torch.empty(n, shape.hidden, dtype=torch.bfloat16, device=DEV),
            "qkv": normal(n, shape.qkv_width), "pos": t, "cos": ang.cos().float(), "sin": ang.sin().float(),
            "kc": kc, "vc": torch.zeros_like(kc), "slots": pool[t // 16] * 16 + t % 16,
            "ks": torch.full((shape.kv_heads,), 4.5 / 127, device=DEV),
            "vs": torch.full((shape.kv_heads,), 4.5 / 127, device=DEV),
            "gate_up": normal(n, 2 * shape.ffn),
            "act": torch.empty(n, shape.ffn, dtype=torch.bfloat16, device=DEV)}


def _step_inputs(case, seed):
    g = _generator(seed)
    shape = decode_loop.QwenShape(layers=case["layers"])
    b, ctx = case["batch"], case["context"]

    def normal(*size, std=0.02):
        return torch.empty(*size, dtype=torch.bfloat16, device=DEV).normal_(0.0, std, generator=g)

    H, D = shape.hidden, shape.head_dim
    layers, caches, scales = [], [], []
    width = decode_loop.blocks_per_sequence(ctx + 1)
    tables = torch.randperm(b * width, generator=g, device=DEV).to(torch.int32).view(b, width)
    for _ in range(shape.layers):
        layers.append({"ln1": normal(H, std=0.1) + 1, "wqkv": normal(shape.qkv_width, H),
                       "bqkv": normal(shape.qkv_width), "wo": normal(H, shape.q_heads * D),
                       "ln2": normal(H, std=0.1) + 1, "w_gate_up": normal(2 * shape.ffn, H),
                       "w_down": normal(H, shape.ffn)})
        mult, offset = _channels(shape.kv_heads, D, g)
        ks, vs = _static_scales(mult, offset, g)
        caches.append(_fill_caches(b * width, 16, mult, offset, case["cache"], ks, vs, g))
        scales.append((ks, vs))
    return {"shape": shape, "layers": layers, "embed": normal(shape.vocab, H, std=1.0),
            "ln_f": normal(H, std=0.1) + 1, "lm_head": normal(shape.vocab, H), "tables": tables,
            "caches": caches, "ks": torch.stack([s[0] for s in scales]),
            "vs": torch.stack([s[1] for s in scales]),
            "tokens": torch.randint(0, shape.vocab, (b,), generator=g, device=DEV)}


def _step_state(case, seed):
    m = _step_inputs(case, seed)
    b, ctx, mode = case["batch"], case["context"], case["cache"]
    weights = decode_loop.ModelWeights(
        shape=m["shape"], embed=m["embed"], ln_f=m["ln_f"], lm_head=m["lm_head"],
        layers=[decode_loop.LayerWeights(**lw) for lw in m["layers"]])
    loop = decode_loop.DecodeLoop(weights, b, ctx, 1, mode,
                                  scales=(m["ks"], m["vs"]) if mode == "int8" else None)
    loop.block_tables.copy_(m["tables"])
    for l, (kc, vc) in enumerate(m["caches"]):
        loop.cache.key[l].copy_(kc)
        loop.cache.value[l].copy_(vc)
    loop.tokens.copy_(m["tokens"])
    loop.positions.fill_(ctx)
    loop.seq_lens.fill_(ctx + 1)
    before = loop.state()
    loop.capture()
    return {"kind": "step", "loop": loop, "before": before}


def prepare(case, seed):
    return {"decode": _decode_inputs, "write": _write_inputs, "prefill_ops": _prefill_inputs,
            "step": _step_state}[case["kind"]](case, seed)


# ------------------------------------------------------------------------------------- passes
def run(s):
    if s["kind"] == "decode":
        if s["append"]:
            int8kv.int8_kv_cache_write(s["new_k"], s["new_v"], s["kc"], s["vc"], s["slots"],
                                       s["ks"], s["vs"])
        if s["cache"] == "int8":
            out = int8kv.int8_paged_attention(s["q"], s["kc"], s["vc"], s["tables"], s["lens"],
                                              s["ks"], s["vs"], quantize_q=s["quantize_q"])
        else:
            out = int8kv.bf16_paged_attention(s["q"], s["kc"], s["vc"], s["tables"], s["lens"])
        return {"out": out, "kc": s["kc"], "vc": s["vc"]} if s["append"] else {"out": out}
    if s["kind"] == "write":
        if s["dynamic"]:
            cache_ops.reshape_and_cache_int8(s["k"], s["v"], s["kc"], s["vc"], s["ksc"], s["vsc"],
                                             s["slots"])
            return {"kc": s["kc"], "vc": s["vc"], "ksc": s["ksc"], "vsc": s["vsc"]}
        int8kv.int8_kv_cache_write(s["k"], s["v"], s["kc"], s["vc"], s["slots"], s["ks"], s["vs"])
        return {"kc": s["kc"], "vc": s["vc"]}
    if s["kind"] == "prefill_ops":
        # The library's calls of one layer of DecodeLoop.prefill, in its order.
        shape = s["shape"]
        heads = shape.q_heads + shape.kv_heads
        decode_loop.hip_rotary_(s["qkv"], heads, shape.head_dim, s["pos"], s["cos"], s["sin"])
        kv = s["qkv"].view(-1, heads + shape.kv_heads, shape.head_dim)
        int8kv.int8_kv_cache_write(kv[:, shape.q_heads:heads], kv[:, heads:], s["kc"], s["vc"],
                                   s["slots"], s["ks"], s["vs"])
        decode_loop.hip_add_rms_norm(s["x"], s["attn_out"], s["w1"], s["h"], shape.rms_eps)
        decode_loop.hip_silu_mul(s["gate_up"], s["act"])
        decode_loop.hip_add_rms_norm(s["x"], s["mlp_out"], s["w2"], s["h2"], shape.rms_eps)
        return {k: s[k] for k in ("qkv", "kc", "vc", "x", "h", "act", "h2")}
    # The step's inputs go into the graph's buffers, as a scheduler puts them there, then the step.
    loop = s["loop"]
    loop.restore(s["before"])
    loop.replay()
    return {"logits": loop.logits, "key": loop.cache.key, "value": loop.cache.value}


# ------------------------------------------------------------------------------------- work
def _decode_bytes(case):
    lens = _lengths(case)
    tokens, blocks = sum(lens), sum(-(-n // case["block"]) for n in lens)
    row = case["hkv"] * case["d"]
    n = (2 * tokens * row * SIZE[case["cache"]] + 4 * blocks + 4 * len(lens)
         + 2 * len(lens) * case["hq"] * case["d"] * SIZE[case["query"]])
    if case["append"]:
        n += len(lens) * (row * 2 * 3 + 8)
    return n


def work(case):
    if case["kind"] == "decode":
        return {"bytes": _decode_bytes(case),
                "flops": 4.0 * sum(_lengths(case)) * case["hq"] * case["d"]}
    if case["kind"] == "write":
        n, row = case["tokens"], case["hkv"] * case["d"]
        scales = 2 * n * case["hkv"] * 4 if case["dynamic"] else 0
        return {"bytes": n * row * 2 * (SIZE[case["source"]] + 1) + scales + 8 * (n + case["padding"]),
                "flops": 0}
    shape = decode_loop.QWEN25_7B
    H, D, F = shape.hidden, shape.head_dim, shape.ffn
    if case["kind"] == "prefill_ops":
        n = case["tokens"]
        rotary = (shape.q_heads + shape.kv_heads) * D * 4 + shape.head_dim * 8  # in and out, tables
        write = shape.kv_heads * D * 2 * 3 + 8
        norms = 2 * H * 2 * 4  # residual in and out, delta, normed
        return {"bytes": n * (rotary + write + norms + 3 * F * 2), "flops": 0}
    b, L = case["batch"], case["layers"]
    per_layer = shape.qkv_width * H + H * shape.q_heads * D + 3 * F * H
    weights = 2 * (L * per_layer + shape.vocab * H)
    kv = 2 * L * b * (case["context"] + 1) * shape.kv_heads * D * SIZE[case["cache"]]
    return {"bytes": weights + kv + 2 * b * shape.vocab,
            "flops": 2.0 * b * (L * per_layer + shape.vocab * H)
            + 4.0 * L * b * (case["context"] + 1) * shape.q_heads * D}


def tolerance(case):
    if case["kind"] == "write":
        return "exact"  # codes, and scales that are one division
    if case["kind"] == "prefill_ops":
        # One bf16 rounding of each result (the sum of squares in another order, exp in another
        # last bit); the codes are of rotated values rounded the same way, and stay the same.
        return {"rel": 4e-3, "max": 3e-2}
    if case["kind"] == "step":
        # bf16 activations through every layer: a flipped rounding travels on (the logits of six
        # layers are 1.5e-2 off those in 64 bits).  Of the caches only the new rows can differ.
        return {"rel": 3e-2, "max": 3e-1, "differ": min(1e-2, 1.0 / (case["context"] + 1))}
    # The output's own rounding dominates for a 16-bit query; fp32 keeps the products' error.
    return {"bf16": {"rel": 5e-3, "max": 3e-2}, "fp16": {"rel": 8e-4, "max": 8e-3},
            "fp32": {"rel": 2e-4, "max": 4e-3}}[case["query"]]


# ------------------------------------------------------------------------------------- exact
def _attention64(q, kc, vc, tables, lens, ks, vs):
    """softmax(q k^T / sqrt(D)) v in 64 bits per sequence; caches as stored, times their scales."""
    b, hq, d = q.shape
    block, hkv = kc.shape[1], kc.shape[2]
    out = torch.zeros(b, hq, d, dtype=torch.float64, device=q.device)
    for i in range(b):
        n = int(lens[i])
        idx = tables[i, : -(-n // block)].long()
        k = kc[idx].reshape(-1, hkv, d)[:n].double().permute(1, 2, 0).contiguous()
        v = vc[idx].reshape(-1, hkv, d)[:n].double().permute(1, 0, 2).contiguous()
        if ks is not None:
            k *= ks.double()[:, None, None]
            v *= vs.double()[:, None, None]
        s = torch.matmul(q[i].double().view(hkv, hq // hkv, d), k) / math.sqrt(d)
        out[i] = torch.matmul(s.softmax(-1), v).view(hq, d)
    return out


def _append64(kc, vc, k, v, ks, vs, slots):
    hkv, d = kc.shape[2:]
    for cache, x, s in ((kc, k, ks), (vc, v, vs)):
        if s is not None:
            x = (x.double() / s.double()[:, None]).round().clamp(-127, 127)
        cache.view(-1, hkv, d)[slots] = x.to(cache.dtype)


def _norm64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rotate64(x, cos, sin):
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos.double().unsqueeze(-2) + turned * sin.double().unsqueeze(-2)


def exact(case, seed):
    if case["kind"] == "decode":
        s = _decode_inputs(case, seed)
        q = s["q"].double()
        if s["append"]:
            _append64(s["kc"], s["vc"], s["new_k"], s["new_v"], s["ks"], s["vs"], s["slots"])
        if s["quantize_q"]:
            qs = (q.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-6)
            r = (q / qs).clamp(-127, 127)
            q = torch.where(r >= 0, (r + 0.5).floor(), (r - 0.5).ceil()) * qs
        int8 = s["cache"] == "int8"
        out = _attention64(q, s["kc"], s["vc"], s["tables"], s["lens"], s["ks"] if int8 else None,
                           s["vs"] if int8 else None)
        return {"out": out, "kc": None, "vc": None} if s["append"] else {"out": out}
    if case["kind"] == "write":
        if not case["dynamic"]:
            return None
        s = _write_inputs(case, seed)
        hkv = case["hkv"]
        ksc, vsc = s["ksc"].double(), s["vsc"].double()
        valid = s["slots"] >= 0
        for cache, x in ((ksc, s["k"]), (vsc, s["v"])):
            cache.view(-1, hkv)[s["slots"][valid]] = (
                x[valid].abs().amax(-1).double() / 127).clamp_min(1e-6)
        return {"kc": None, "vc": None, "ksc": ksc, "vsc": vsc}
    if case["kind"] == "prefill_ops":
        s = _prefill_inputs(case, seed)
        shape = s["shape"]
        heads = shape.q_heads + shape.kv_heads
        qkv = s["qkv"].double().view(-1, heads + shape.kv_heads, shape.head_dim)
        qkv[:, :heads] = _rotate64(qkv[:, :heads].clone(), s["cos"], s["sin"])
        x1 = s["x"].double() + s["attn_out"].double()
        x2 = x1 + s["mlp_out"].double()
        gate, up = s["gate_up"].double().split(shape.ffn, dim=1)
        return {"qkv": qkv.view_as(s["qkv"]), "kc": None, "vc": None, "x": x2,
                "h": _norm64(x1, s["w1"], shape.rms_eps), "act": torch.nn.functional.silu(gate) * up,
                "h2": _norm64(x2, s["w2"], shape.rms_eps)}
    m = _step_inputs(case, seed)
    shape, b, ctx = m["shape"], case["batch"], case["context"]
    Hq, Hkv, D = shape.q_heads, shape.kv_heads, shape.head_dim
    int8 = case["cache"] == "int8"
    half = D // 2
    freq = shape.rope_theta ** (torch.arange(half, dtype=torch.float64, device=DEV) * -2.0 / D)
    ang = (freq * ctx).repeat(2)[None, :]
    slots = m["tables"][:, ctx // 16].long() * 16 + ctx % 16
    lens = [ctx + 1] * b
    x = m["embed"][m["tokens"]].double()
    for l, lw in enumerate(m["layers"]):
        h = _norm64(x, lw["ln1"], shape.rms_eps)
        qkv = (h @ lw["wqkv"].double().t() + lw["bqkv"].double()).view(b, Hq + 2 * Hkv, D)
        qk = _rotate64(qkv[:, : Hq + Hkv], ang.cos(), ang.sin())
        kc, vc = m["caches"][l]
        ks, vs = (m["ks"][l], m["vs"][l]) if int8 else (None, None)
        _append64(kc, vc, qk[:, Hq:], qkv[:, Hq + Hkv:], ks, vs, slots)
        attn = _attention64(qk[:, :Hq], kc, vc, m["tables"], lens, ks, vs).view(b, Hq * D)
        x = x + attn @ lw["wo"].double().t()
        gu = _norm64(x, lw["ln2"], shape.rms_eps) @ lw["w_gate_up"].double().t()
        gate, up = gu.split(shape.ffn, dim=1)
        x = x + (torch.nn.functional.silu(gate) * up) @ lw["w_down"].double().t()
    h = _norm64(x, m["ln_f"], shape.rms_eps)
    return {"logits": h @ m["lm_head"].double().t(), "key": None, "value": None}
