"""Performance cases of the attention path: the calls a serving program makes per layer and step.

A case is a dict of plain values; `prepare` builds what such a program holds before the
call (tensors, bound caches, captured graphs), `run` makes one pass through the public
entry points and returns its outputs (the attention output and the caches it stored to),
`work` counts the bytes and operations the pass cannot do without, and `exact` restates it
in float64 with plain torch.  Kinds:
  decode    Attention.forward of one layer in a decode step (store of the new token, then
            paged attention over the context), eager
  graph     DecodeGraphs.run: the attention path of all layers as one captured step
  prefill   Attention.forward of one layer over fresh prompt tokens, after a cached prefix
            (read through the block table) when `prefix_pages` is not 0
  producer  qk_norm_rope: per-head RMSNorm (Qwen3) and rotary embedding of q and k

Sequence lengths are `batch` draws of U[lo, hi] from `lens_seed`, so the work of a case does
not depend on the seed of its values.  Pages hold 256 tokens, the default of the engine.
"""
from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parents[1] / "nano-vllm_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

import nanovllm_amd as nva  # noqa: E402
from nanovllm_amd import workloads as W  # noqa: E402
from nanovllm_amd.engine.decode_graphs import DecodeGraphs  # noqa: E402
from nanovllm_amd.layers.qk_norm_rope import qk_norm_rope  # noqa: E402

PAGE = 256
FP8 = torch.float8_e4m3fn
# A decode graph's table is sized for 4096 tokens, the default max_model_len.
GRAPH_BLOCKS = 16
# Query heads, kv heads and head dim of the shapes served: Qwen3-0.6B, -8B, -32B, the last
# two as one GPU's share of eight, and Qwen2-0.5B.
HEADS = [(16, 8, 128), (32, 8, 128), (64, 8, 128), (4, 1, 128), (8, 1, 128), (14, 2, 64)]


def _decode(nh, nkv, d, batch, lo, hi, lens_seed, fp8=False):
    return {"kind": "decode", "nh": nh, "nkv": nkv, "d": d, "batch": batch, "lo": lo, "hi": hi,
            "lens_seed": lens_seed, "fp8": fp8}


def _graph(nh, nkv, d, layers, batch, lo, hi, lens_seed):
    return {"kind": "graph", "nh": nh, "nkv": nkv, "d": d, "layers": layers, "batch": batch, "lo": lo, "hi": hi,
            "lens_seed": lens_seed}


def _prefill(nh, nkv, d, batch, lo, hi, lens_seed, prefix_pages=0, shared=False, fp8=False):
    return {"kind": "prefill", "nh": nh, "nkv": nkv, "d": d, "batch": batch, "lo": lo, "hi": hi,
            "lens_seed": lens_seed, "prefix_pages": prefix_pages, "shared": shared, "fp8": fp8}


def _producer(nh, nkv, d, tokens, norm):
    return {"kind": "producer", "nh": nh, "nkv": nkv, "d": d, "tokens": tokens, "norm": norm}


def listed():
    def named(name, case):
        return {"name": name, **case}
    return [
        # one interactive user: a single sequence, where only latency counts
        named("decode_one", _decode(16, 8, 128, 1, 517, 517, 1)),
        # a few users of the small model (7 query heads per kv head, head dim 64)
        named("decode_small_d64", _decode(14, 2, 64, 8, 100, 2048, 2)),
        # a service at moderate load: an odd batch of ragged contexts, 8B heads
        named("decode_mid", _decode(32, 8, 128, 37, 256, 4096, 3)),
        # the throughput benchmark's decode step: 256 sequences of 100 to 2048 tokens
        named("decode_batch", _decode(16, 8, 128, 256, 100, 2048, 1003)),
        # long contexts over the fp8 cache, 32B heads: the largest decode
        named("decode_fp8_long", _decode(64, 8, 128, 64, 16384, 32768, 1005, fp8=True)),
        # the captured decode step of all 28 layers, 13 rows in the graph of 16
        named("graph_decode", _graph(16, 8, 128, 28, 13, 100, 2048, 4)),
        # eight short prompts without a cached prefix
        named("prefill_short", _prefill(16, 8, 128, 8, 100, 1024, 1002)),
        # sixteen prompts behind a shared 1024-token prefix (a system prompt), 8B heads
        named("prefill_prefix", _prefill(32, 8, 128, 16, 256, 768, 1004, prefix_pages=4, shared=True)),
        # continued conversations over the fp8 cache: each sequence has its own cached pages
        named("prefill_prefix_fp8", _prefill(32, 8, 128, 6, 100, 1500, 5, prefix_pages=6, fp8=True)),
        # one long document, nearly the 16384 tokens that a batch may hold
        named("prefill_long", _prefill(16, 8, 128, 1, 16001, 16001, 6)),
        # prompts of the small model, head dim 64
        named("prefill_d64", _prefill(14, 2, 64, 12, 100, 1024, 7)),
        # qk-norm and rotary embedding of a prompt batch, 8B heads
        named("producer", _producer(32, 8, 128, 8813, True)),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 4 + ["producer", "graph"])
    nh, nkv, d = rng.choice(HEADS)
    seed = rng.randrange(1 << 30)
    if kind == "producer":
        return _producer(nh, nkv, d, _log_int(rng, 1, 16384), d == 128)
    if kind == "graph":
        layers = rng.randint(4, 28)
        hi = _log_int(rng, 32, GRAPH_BLOCKS * PAGE)
        # at most about 1.5 GB of keys and values per step
        most = max(1, int(1.5e9 / (layers * hi * nkv * d * 4)))
        return _graph(nh, nkv, d, layers, _log_int(rng, 1, min(64, most)), max(1, hi // 8), hi, seed)
    if kind == "decode":
        fp8 = d == 128 and rng.random() < 0.35
        hi = _log_int(rng, 16, 32768)
        most = max(1, int(3e9 / (hi * nkv * d * (2 if fp8 else 4))))
        return _decode(nh, nkv, d, _log_int(rng, 1, min(256, most)), max(1, hi // rng.choice([1, 2, 16])), hi, seed, fp8)
    hi = _log_int(rng, 8, 16384)
    pages = rng.choice([0, 0, 1, 4, 8])
    # at most 16384 new tokens, and the operations of the longest listed prompt
    most = min(16384 // hi, int(1.0e12 / (4 * d * nh * hi * (hi / 2 + pages * PAGE))))
    if most < 1:
        nh, nkv, d, pages, most = 16, 8, 128, 0, 1
    fp8 = bool(pages) and d == 128 and rng.random() < 0.5
    return _prefill(nh, nkv, d, _log_int(rng, 1, min(64, most)), max(1, hi // rng.choice([1, 2, 8])), hi, seed,
                    pages, bool(pages) and rng.random() < 0.5, fp8)


def _lens(case):
    g = torch.Generator().manual_seed(case["lens_seed"])
    return torch.randint(case["lo"], case["hi"] + 1, (case["batch"],), generator=g).tolist()


def _pages(n):
    return -(-n // PAGE)


def _layer(case, k_cache, v_cache, k_scale=None, v_scale=None):
    layer = nva.Attention(case["nh"], case["d"], case["d"] ** -0.5, case["nkv"])
    layer.k_cache, layer.v_cache, layer.k_scale, layer.v_scale = k_cache, v_cache, k_scale, v_scale
    return layer


def prepare(case, seed):
    dev, kind = torch.device("cuda"), case["kind"]
    nh, nkv, d = case["nh"], case["nkv"], case["d"]
    if kind == "producer":
        return {"case": case, "in": W.make_producer_case(case["tokens"], nh, nkv, head_dim=d, norm=case["norm"],
                                                         seed=seed, device=dev)}
    lens = _lens(case)
    if kind == "prefill":
        prefix, blocks = case["prefix_pages"] * PAGE, sum(_pages(n) for n in lens)
        blocks += case["prefix_pages"] * (1 if case["shared"] else len(lens))
        c = W.make_prefill_case(lens, nh, nkv, blocks, prefix_len=prefix, head_dim=d, seed=seed, bulk_device=dev,
                                shared_prefix=case["shared"])
        scales = (None, None)
        if case["fp8"]:
            c.k_cache, ks = W.quantize_cache_fp8(c.k_cache, extra=c.k)
            c.v_cache, vs = W.quantize_cache_fp8(c.v_cache, extra=c.v)
            scales = (ks, vs)
        return {"case": case, "in": c, "layer": _layer(case, c.k_cache, c.v_cache, *scales)}
    blocks = sum(_pages(n) for n in lens)
    c = W.make_decode_case(case["batch"], nh, nkv, 0, 0, blocks, head_dim=d, fp8=case.get("fp8", False), seed=seed,
                           bulk_device=dev, lengths=lens)
    if kind == "decode":
        return {"case": case, "in": c, "layer": _layer(case, c.k_cache, c.v_cache, c.k_scale, c.v_scale)}
    g = torch.Generator(device=dev).manual_seed(seed + 1)
    kv = torch.empty(2, case["layers"], blocks, PAGE, nkv, d, dtype=torch.bfloat16, device=dev)
    for side in kv:
        for one in side:
            one.normal_(generator=g)
    layers = [_layer(case, kv[0, i], kv[1, i]) for i in range(case["layers"])]
    sizes = -(-case["batch"] // 16) * 16
    return {"case": case, "in": c, "kv": kv, "graphs": DecodeGraphs(layers, sizes, GRAPH_BLOCKS).capture()}


def _cache_bytes(t):
    """The cache's stored values as whole numbers: a store copies or quantises them bit for bit."""
    return t.view(torch.int16 if t.dtype == torch.bfloat16 else torch.uint8)


def run(state):
    case, c = state["case"], state["in"]
    kind = case["kind"]
    if kind == "producer":
        q, k = qk_norm_rope(c.positions, c.q, c.k, c.cos_sin_cache, c.num_heads, c.num_kv_heads, c.head_dim,
                            c.q_norm_weight, c.k_norm_weight, c.eps)
        return {"q": q, "k": k}
    if kind == "graph":
        outs = state["graphs"].run(c.q, c.k_new, c.v_new, c.slot_mapping, c.context_lens, c.block_tables)
        return {"o": outs, "kv": _cache_bytes(state["kv"])}
    layer = state["layer"]
    if kind == "prefill":
        nva.set_context(True, c.cu_seqlens_q, c.cu_seqlens_k, c.max_seqlen_q, c.max_seqlen_k, c.slot_mapping, None,
                        c.block_tables)
        o = layer(c.q, c.k, c.v)
    else:
        nva.set_context(False, slot_mapping=c.slot_mapping, context_lens=c.context_lens, block_tables=c.block_tables)
        o = layer(c.q, c.k_new, c.v_new)
    nva.reset_context()
    return {"o": o, "k_cache": _cache_bytes(layer.k_cache), "v_cache": _cache_bytes(layer.v_cache)}


def work(case):
    kind, nh, nkv, d = case["kind"], case["nh"], case["nkv"], case["d"]
    if kind == "producer":
        t = case["tokens"]
        return {"bytes": t * ((nh + nkv) * d * 4 + d * 4 + 8), "flops": t * (nh + nkv) * d * (8 if case["norm"] else 3)}
    lens = _lens(case)
    elem = 1 if case.get("fp8") else 2
    if kind == "prefill":
        pre = case["prefix_pages"] * PAGE
        pairs = sum(n * pre + n * (n + 1) // 2 for n in lens)
        t = sum(lens)
        cached = pre * (1 if case["shared"] else len(lens))
        return {"bytes": 2 * t * nh * d * 2 + 2 * t * nkv * d * (2 + elem) + 2 * cached * nkv * d * elem + 4 * t,
                "flops": 4 * d * nh * pairs}
    # a decode step reads every cached key and value, the new token's, q and the index
    # tensors, and writes the output and the new token's cache rows
    n, b = sum(lens), case["batch"]
    one = 2 * (n - b) * nkv * d * elem + 2 * b * nkv * d * (2 + elem) + 2 * b * nh * d * 2 + 4 * sum(_pages(x) for x in lens)
    layers = case.get("layers", 1)
    return {"bytes": layers * one, "flops": layers * 4 * d * nh * n}


def tolerance(case):
    # bf16 outputs (and, in prefill, bf16 probabilities) against float64; the cache bytes
    # (and whole values in general) have to be the same
    return {"rel": 0.01, "max": 0.06}


def _attend(q, k, v, scale, rows=1024):
    """Causal attention, bottom-right aligned, of q (n, nh, d) over k, v (m, nkv, d), float64."""
    n, nh, d = q.shape
    m, nkv = k.shape[:2]
    g = nh // nkv
    out = torch.empty(n, nh, d, dtype=torch.float64, device=q.device)
    kt, vt = k.double().permute(1, 2, 0).contiguous(), v.double().permute(1, 0, 2).contiguous()
    key = torch.arange(m, device=q.device)
    for i in range(0, n, rows):
        r = q[i:i + rows].double()
        t = r.shape[0]
        see = i + t + m - n  # keys visible to the chunk's last row
        r = r.view(t, nkv, g, d).permute(1, 2, 0, 3).reshape(nkv, g * t, d)
        s = torch.bmm(r, kt[:, :, :see].contiguous()).view(nkv, g, t, see) * scale
        last = torch.arange(i, i + t, device=q.device) + (m - n)
        s.masked_fill_(key[None, :see] > last[:, None], -math.inf)
        p = torch.softmax(s, -1).view(nkv, g * t, see)
        o = torch.bmm(p, vt[:, :see].contiguous()).view(nkv, g, t, d)
        out[i:i + t] = o.permute(2, 0, 1, 3).reshape(t, nh, d)
    return out


def _stored(cache, new, slots, scale):
    """(slots, nkv, d) view of the cache's values after `new` went to `slots`, and its scale per head."""
    flat = cache.view(-1, *cache.shape[2:]).clone()
    if flat.dtype == FP8:
        new = (new.float() / scale.view(1, -1, 1)).to(FP8)
        flat.view(torch.uint8)[slots.long()] = new.view(torch.uint8)
        return flat, scale.double().view(1, -1, 1)
    flat[slots.long()] = new
    return flat, 1.0


def _rows(stored, table, n):
    flat, scale = stored
    pages = table[:_pages(n)].long()
    at = (pages[:, None] * PAGE + torch.arange(PAGE, device=table.device)).view(-1)[:n]
    x = flat.view(torch.uint8)[at].view(FP8) if flat.dtype == FP8 else flat[at]
    return x.float().double() * scale


def _decode64(c, k_cache, v_cache, k_scale=None, v_scale=None):
    ks, vs = (_stored(t, x, c.slot_mapping, s) for t, x, s in ((k_cache, c.k_new, k_scale), (v_cache, c.v_new, v_scale)))
    rows = [_attend(c.q[b:b + 1], _rows(ks, c.block_tables[b], n), _rows(vs, c.block_tables[b], n), c.scale)
            for b, n in enumerate(c.lengths)]
    return torch.cat(rows).view(len(rows), -1)


def exact(case, seed):
    state = prepare({**case, "kind": "decode"} if case["kind"] == "graph" else case, seed)
    kind, c = case["kind"], state["in"]
    if kind == "producer":
        cs = c.cos_sin_cache[c.positions].double()
        cos, sin = cs[:, None, :c.head_dim // 2], cs[:, None, c.head_dim // 2:]

        def one(x, w):
            x = x.double()
            if w is not None:
                x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + c.eps) * w.double()
            a, b = x.chunk(2, -1)
            return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)
        return {"q": one(c.q, c.q_norm_weight), "k": one(c.k, c.k_norm_weight)}
    if kind == "graph":
        dev = c.q.device
        g = torch.Generator(device=dev).manual_seed(seed + 1)
        kv = torch.empty(2, case["layers"], *c.k_cache.shape, dtype=torch.bfloat16, device=dev)
        for side in kv:
            for one in side:
                one.normal_(generator=g)
        return {"o": [_decode64(c, kv[0, i], kv[1, i]) for i in range(case["layers"])], "kv": None}
    layer = state["layer"]
    if kind == "decode":
        return {"o": _decode64(c, layer.k_cache, layer.v_cache, layer.k_scale, layer.v_scale), "k_cache": None,
                "v_cache": None}
    k = (layer.k_cache, c.k, layer.k_scale)
    v = (layer.v_cache, c.v, layer.v_scale)
    if c.block_tables is not None:
        ks, vs = (_stored(t, x, c.slot_mapping, s) for t, x, s in (k, v))
    rows, at = [], 0
    for s, (n, m) in enumerate(zip(c.lens_q, c.lens_k)):
        if c.block_tables is not None:
            kk, vv = _rows(ks, c.block_tables[s], m), _rows(vs, c.block_tables[s], m)
        else:
            kk, vv = c.k[at:at + n], c.v[at:at + n]
        rows.append(_attend(c.q[at:at + n], kk, vv, c.scale))
        at += n
    return {"o": torch.cat(rows).view(at, -1), "k_cache": None, "v_cache": None}
