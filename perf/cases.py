"""Performance cases of the KV-cache compression path: what a serving engine, a HuggingFace prefill hook and a cache
quantiser ask of this package, through the entry points they call.

``kind`` of a case:

``press-hook``    ``KnormPress`` / ``SnapKVPress`` ``.compress`` on one layer's ``[B, Hkv, S, D]`` tensors, what the press's
                  forward hook runs for every attention layer of a prefill
``press-runner``  the same presses as the compressor of a ``PagedKVRunner``: ``compress_kv_cache_batch`` over all layers
                  of a batch of sequences, in place in the page pool
``ccm-forward``   an MLP compressor module called on a per-layer list of dense tensors
``ccm-runner``    the same compressors on the runner, in place in the pages
``decode``        one decode step over the paged caches: ``prepare_decode``, then every attention layer, called one by
                  one or replayed from the captured graph of the batch's bucket
``quant``         ``QuantizationMethod``: codes and scales of one layer's K and V, then back to values

The in-place kinds hand out the page pool.  A press moves rows and computes none, so its rows are handed out as
whole numbers (``view`` on the same bytes).
"""
from __future__ import annotations

import random
from collections import deque
from types import SimpleNamespace

import torch

from fastcache_amd.autocompress.methods import QuantizationMethod
from fastcache_amd.engine.block_manager import BlockManager
from fastcache_amd.engine.decode_graph import BucketedDecodeGraphs
from fastcache_amd.engine.kv_runner import PagedKVRunner
from fastcache_amd.engine.sequence import Sequence
from fastcache_amd.layers.attention import Attention
from fastcache_amd.presses import KnormPress, SnapKVPress
from fastcache_amd.utils_ccm import KVCacheHybridCompressor, KVCacheLinearDecoupleCompressor

D = 128                # head dimension of every model this package serves
PAGE = 256             # tokens per page
_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # a short chat prompt through the Knorm hook: one layer, a handful of small launches
        {"name": "hook-knorm-short", "kind": "press-hook", "press": "knorm", "dtype": "bf16", "batch": 1, "q_heads": 32,
         "kv_heads": 8, "seq_len": 333, "ratio": 0.5, "window": 0},
        # a batch of 4k prompts through the SnapKV hook, one layer at a time, the press's default window and pooling
        {"name": "hook-snapkv-4k", "kind": "press-hook", "press": "snapkv", "dtype": "bf16", "batch": 4, "q_heads": 32,
         "kv_heads": 8, "seq_len": 4096, "ratio": 0.5, "window": 64},
        # benchmark configuration 1: one LLaMA-7B-shaped fp32 prompt, half of it kept
        {"name": "runner-knorm-fp32", "kind": "press-runner", "press": "knorm", "dtype": "f32", "layers": 32, "batch": 1,
         "q_heads": 32, "kv_heads": 32, "min_len": 1024, "max_len": 1024, "ratio": 0.5, "window": 0, "lens_seed": 0},
        # benchmark configuration 2: eight Qwen3-8B-shaped prompts of 4k, a quarter kept
        {"name": "runner-snapkv-4k", "kind": "press-runner", "press": "snapkv", "dtype": "bf16", "layers": 36, "batch": 8,
         "q_heads": 32, "kv_heads": 8, "min_len": 4096, "max_len": 4096, "ratio": 0.75, "window": 64, "lens_seed": 0},
        # the lazy trigger: whatever is running when pages run short, every sequence of another length
        {"name": "runner-snapkv-ragged", "kind": "press-runner", "press": "snapkv", "dtype": "f16", "layers": 28,
         "batch": 13, "q_heads": 28, "kv_heads": 4, "min_len": 200, "max_len": 2300, "ratio": 0.6, "window": 32,
         "lens_seed": 1},
        # one long document: few columns of many keys
        {"name": "runner-snapkv-30k", "kind": "press-runner", "press": "snapkv", "dtype": "bf16", "layers": 36, "batch": 1,
         "q_heads": 32, "kv_heads": 8, "min_len": 30011, "max_len": 30011, "ratio": 0.8, "window": 64, "lens_seed": 0},
        # one image prompt (576 image tokens and a short question) through the compressor module of a HuggingFace script
        {"name": "ccm-forward-one-prompt", "kind": "ccm-forward", "model": "decouple", "dtype": "f16", "layers": 32,
         "batch": 1, "kv_heads": 32, "image_len": 576, "text_len": 47, "factor": 2},
        # benchmark configuration 3: a batch of 45 such prompts on the runner
        {"name": "runner-ccm-batch-45", "kind": "ccm-runner", "model": "decouple", "dtype": "f16", "layers": 32, "batch": 45,
         "kv_heads": 32, "image_len": 576, "min_len": 640, "max_len": 640, "factor": 2, "lens_seed": 0},
        # benchmark configuration 5: long MiniCPM-V-2.6-shaped prompts compressed to a fifth
        {"name": "runner-hybrid-16k", "kind": "ccm-runner", "model": "hybrid", "dtype": "bf16", "layers": 28, "batch": 16,
         "kv_heads": 4, "image_len": 0, "min_len": 16384, "max_len": 16384, "factor": 5, "lens_seed": 0},
        # three users, layers called one by one from Python: launches and host work
        {"name": "decode-eager-3", "kind": "decode", "graph": False, "dtype": "bf16", "layers": 28, "batch": 3,
         "q_heads": 28, "kv_heads": 4, "min_len": 300, "max_len": 900, "lens_seed": 2},
        # benchmark configuration 4 by the bucketed graphs of the reference's protocol: 90 compressed caches
        {"name": "decode-graph-90", "kind": "decode", "graph": True, "dtype": "f16", "layers": 16, "batch": 90,
         "q_heads": 32, "kv_heads": 32, "min_len": 128, "max_len": 2048, "lens_seed": 3},
        # int8 rows of one layer's cache, there and back
        {"name": "quant-int8-layer", "kind": "quant", "type": "int8", "dtype": "bf16", "batch": 8, "kv_heads": 8,
         "seq_len": 4096},
    ]


# ---------------------------------------------------------------------------------------------------------------------
# more of the same ranges
# ---------------------------------------------------------------------------------------------------------------------
def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _batch(rng, lo, hi, budget):
    """A batch size whose total (``budget`` = what one unit may be multiplied with) stays below the largest case."""
    return max(1, min(_log(rng, lo, hi), int(budget)))


def draw(rng):
    kind = rng.choice(["press-hook", "press-runner", "press-runner", "ccm-forward", "ccm-runner", "decode", "decode", "quant"])
    half = rng.choice(["f16", "bf16"])
    if kind == "press-hook":
        press = rng.choice(["knorm", "snapkv"])
        hq, hkv = rng.choice([(32, 8), (28, 4), (32, 32)])
        s = _log(rng, 200, 12000)
        return {"kind": kind, "press": press, "dtype": half, "batch": _batch(rng, 1, 8, 65536 // s), "q_heads": hq,
                "kv_heads": hkv, "seq_len": s, "ratio": rng.choice([0.3, 0.5, 0.75, 0.8]),
                "window": rng.choice([32, 64]) if press == "snapkv" else 0}
    if kind == "press-runner":
        press = rng.choice(["knorm", "snapkv"])
        layers, hq, hkv = rng.choice([(36, 32, 8), (28, 28, 4), (32, 32, 32)])
        hi = _log(rng, 300, 30000 if hkv < 32 else 4000)
        ragged = rng.random() < 0.5
        return {"kind": kind, "press": press, "dtype": rng.choice(["f32", half]) if press == "knorm" else half,
                "layers": layers, "batch": _batch(rng, 1, 16, 9_000_000 // (layers * hkv * hi)), "q_heads": hq,
                "kv_heads": hkv, "min_len": max(150, hi // 8) if ragged else hi, "max_len": hi,
                "ratio": rng.choice([0.3, 0.5, 0.6, 0.75, 0.8]), "window": rng.choice([32, 64]) if press == "snapkv" else 0,
                "lens_seed": rng.randrange(1000)}
    if kind == "ccm-forward":
        model = rng.choice(["decouple", "hybrid"])
        text = _log(rng, 20, 1500)
        return {"kind": kind, "model": model, "dtype": half, "layers": 32 if model == "decouple" else 28,
                "batch": _log(rng, 1, 8), "kv_heads": 32 if model == "decouple" else 4,
                "image_len": 576 if model == "decouple" else 0, "text_len": text if model == "decouple" else 4 * text,
                "factor": rng.choice([2, 5])}
    if kind == "ccm-runner":
        model = rng.choice(["decouple", "hybrid"])
        if model == "decouple":
            hi = 576 + _log(rng, 20, 1000)
            return {"kind": kind, "model": model, "dtype": half, "layers": 32, "batch": _batch(rng, 1, 45, 28800 // hi),
                    "kv_heads": 32, "image_len": 576, "min_len": rng.choice([hi, 590]), "max_len": hi,
                    "factor": rng.choice([2, 5]), "lens_seed": rng.randrange(1000)}
        hi = _log(rng, 700, 16384)
        return {"kind": kind, "model": model, "dtype": half, "layers": 28, "batch": _batch(rng, 1, 16, 262144 // hi),
                "kv_heads": 4, "image_len": 0, "min_len": rng.choice([hi, hi // 3]), "max_len": hi,
                "factor": rng.choice([2, 5]), "lens_seed": rng.randrange(1000)}
    if kind == "decode":
        hq, hkv = rng.choice([(32, 32), (32, 8), (28, 4)])
        hi = _log(rng, 200, 8000)
        graph = rng.random() < 0.6
        return {"kind": kind, "graph": graph, "dtype": half, "layers": rng.choice([8, 12, 16]) if graph else 28,
                "batch": _batch(rng, 1, 90 if graph else 12, 3_000_000 // (hi * hkv)), "q_heads": hq, "kv_heads": hkv,
                "min_len": max(100, hi // 10), "max_len": hi, "lens_seed": rng.randrange(1000)}
    s = _log(rng, 300, 16000)
    return {"kind": kind, "type": rng.choice(["int8", "int4", "nf4", "fp8"]), "dtype": half,
            "batch": _batch(rng, 1, 16, 131072 // s), "kv_heads": rng.choice([4, 8, 32]), "seq_len": s}


# ---------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------
def _lens(case):
    lo, hi = case["min_len"], case["max_len"]
    r = random.Random(case["lens_seed"])
    lens = [r.randint(lo, hi) for _ in range(case["batch"])]
    lens[r.randrange(len(lens))] = hi
    return lens


def _normal(shape, dtype, g):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=g)


def _outlier_channels(keys, g):
    """Keys of trained models have a few channels per head far above the rest: four of them, scaled by 8."""
    H = keys.shape[-2]
    which = torch.rand((H, D), generator=g, device="cuda").argsort(1)[:, :4]
    keys *= torch.ones((H, D), device="cuda").scatter_(1, which, 8.0).to(keys.dtype)


def _paged(case, g, seed, extra_tokens=0, **runner):
    """A pool, its page manager and the sequences of the case, on pages scattered over the pool."""
    lens = _lens(case)
    pages = sum(-(-(n + extra_tokens) // PAGE) for n in lens) + 2
    pool = _normal((2, case["layers"], pages, PAGE, case["kv_heads"], D), _DTYPES[case["dtype"]], g)
    manager = BlockManager(pages, PAGE)
    order = list(range(pages))
    random.Random(seed).shuffle(order)
    manager.free_block_ids = deque(order)
    seqs = []
    for b, n in enumerate(lens):
        s = Sequence(range(b * 100_000, b * 100_000 + n))
        manager.allocate(s)
        while len(s.block_table) * PAGE < n + extra_tokens:
            s.block_table.append(manager._claim_next().block_id)
        seqs.append(s)
    return PagedKVRunner.adopt(pool, block_manager=manager, **runner), seqs, lens


def _press(case):
    if case["press"] == "knorm":
        return KnormPress(case["ratio"])
    return SnapKVPress(case["ratio"], window_size=case["window"], kernel_size=7 if case["kind"] == "press-runner" else 5)


def _compressor(case, seed):
    L, H = case["layers"], case["kv_heads"]
    torch.manual_seed(seed)
    if case["model"] == "decouple":
        cfg = SimpleNamespace(text_config=SimpleNamespace(num_hidden_layers=L, num_key_value_heads=H, hidden_size=H * D))
        module = KVCacheLinearDecoupleCompressor(cfg, compression_factor=case["factor"])
    else:
        cfg = SimpleNamespace(architectures=["MiniCPMV"], num_hidden_layers=L, num_key_value_heads=H,
                              num_attention_heads=7 * H, hidden_size=7 * H * D)
        module = KVCacheHybridCompressor(cfg, compression_factor=case["factor"])
    return module.to(device="cuda", dtype=_DTYPES[case["dtype"]]).eval()


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, dt = case["kind"], _DTYPES[case["dtype"]]
    s = SimpleNamespace(kind=kind, case=case)
    if kind == "press-hook":
        B, H, S = case["batch"], case["kv_heads"], case["seq_len"]
        # what a prefill's attention layer leaves in the cache
        s.keys, s.values = _normal((B, S, H, D), dt, g), _normal((B, S, H, D), dt, g)
        if case["press"] == "knorm":
            _outlier_channels(s.keys, g)
        s.keys, s.values = s.keys.transpose(1, 2).contiguous(), s.values.transpose(1, 2).contiguous()
        s.hidden = torch.zeros((B, S, 1), dtype=dt, device="cuda")       # of which these presses read only the length
        s.kwargs = {}
        if case["press"] == "snapkv":
            s.kwargs["queries"] = _normal((B, case["q_heads"], case["window"], D), dt, g)
        s.press = _press(case)
    elif kind == "press-runner":
        s.press = _press(case)
        s.runner, s.seqs, _ = _paged(case, g, seed, compressor=s.press, image_token_len=0)
        s.queries = None
        if case["press"] == "knorm":
            _outlier_channels(s.runner.kv_cache[0], g)
        else:
            s.queries = _normal((case["layers"], case["batch"], case["q_heads"], case["window"], D), dt, g)
    elif kind == "ccm-forward":
        S = case["image_len"] + case["text_len"]
        shape = (case["batch"], case["kv_heads"], S, D)
        s.module = _compressor(case, seed)
        s.cache = [(_normal(shape, dt, g), _normal(shape, dt, g)) for _ in range(case["layers"])]
        s.it_len = [case["image_len"], case["text_len"]]
    elif kind == "ccm-runner":
        s.runner, s.seqs, _ = _paged(case, g, seed, compressor=_compressor(case, seed), image_token_len=case["image_len"])
    elif kind == "decode":
        L, B, hq, hkv = case["layers"], case["batch"], case["q_heads"], case["kv_heads"]
        s.runner, s.seqs, lens = _paged(case, g, seed, extra_tokens=1)
        s.layers = [Attention(hq, D, D ** -0.5, hkv) for _ in range(L)]
        for i, layer in enumerate(s.layers):
            layer.k_cache, layer.v_cache = s.runner.kv_cache[0, i], s.runner.kv_cache[1, i]
        s.q, s.k, s.v = (_normal((L, B, h * D), dt, g) for h in (hq, hkv, hkv))
        s.graphs = None
        if case["graph"]:
            s.graphs = BucketedDecodeGraphs(s.layers, B, max(n // PAGE + 1 for n in lens), dt, "cuda")
            s.graphs.capture_cudagraph()
    else:
        shape = (case["batch"], case["kv_heads"], case["seq_len"], D)
        s.method = QuantizationMethod(case["type"])
        s.keys, s.values = _normal(shape, dt, g), _normal(shape, dt, g)
        s.dtype = dt
    return s


def _as_whole(t):
    return t.view(torch.int32 if t.element_size() == 4 else torch.int16)


def run(s):
    if s.kind == "press-hook":
        k, v = s.press.compress(None, s.hidden, s.keys, s.values, None, s.kwargs)
        return _as_whole(k), _as_whole(v)
    if s.kind == "press-runner":
        if s.queries is not None:
            s.press.set_window_queries(s.queries, seq_ids=[q.seq_id for q in s.seqs])
        _, ratio = s.runner.compress_kv_cache_batch(s.seqs)
        return _as_whole(s.runner.kv_cache), ratio
    if s.kind == "ccm-forward":
        return s.module(s.cache, s.it_len)
    if s.kind == "ccm-runner":
        _, ratio = s.runner.compress_kv_cache_batch(s.seqs)
        return s.runner.kv_cache, ratio
    if s.kind == "decode":
        s.runner.prepare_decode(s.seqs)
        if s.graphs is not None:
            out = s.graphs.run(s.q, s.k, s.v)
        else:
            out = [layer(s.q[i], s.k[i], s.v[i]) for i, layer in enumerate(s.layers)]
        return {"out": out, "k_cache": s.runner.kv_cache[0], "v_cache": s.runner.kv_cache[1]}
    (qk, sk), (qv, sv) = s.method.compress(s.keys, s.values)
    back = [s.method.dequantize(qk, sk, s.dtype), s.method.dequantize(qv, sv, s.dtype)]
    return {"codes": [qk.view(torch.uint8), qv.view(torch.uint8)], "scales": [sk, sv], "back": back}


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def _segment(n, cf):
    """(rows through the MLP, rows copied behind them) of a segment of n tokens."""
    return (n // cf, n % cf) if n // cf >= 1 else (0, n)


def work(case):
    kind, e = case["kind"], _BYTES[case["dtype"]]
    row = D * e
    if kind in ("press-hook", "press-runner"):
        layers = case.get("layers", 1)
        lens = _lens(case) if kind == "press-runner" else [case["seq_len"]] * case["batch"]
        kept = [int(n * (1 - case["ratio"])) for n in lens]
        cols = layers * case["kv_heads"]
        # every key once for its score, the kept values once, the kept rows of both written
        nbytes = cols * row * (sum(lens) + 3 * sum(kept)) + layers * len(lens) * case["q_heads"] * case["window"] * row
        flops = 2 * layers * case["q_heads"] * case["window"] * D * sum(lens) if case["window"] else 2 * cols * D * sum(lens)
        return {"bytes": nbytes, "flops": flops}
    if kind in ("ccm-forward", "ccm-runner"):
        cf, cols = case["factor"], 2 * case["layers"] * case["kv_heads"]
        lens = _lens(case) if kind == "ccm-runner" else [case["image_len"] + case["text_len"]] * case["batch"]
        rows = copied = 0
        for n in lens:
            img = min(case["image_len"], n)
            for part in (img, n - img):
                r, c = _segment(part, cf)
                rows, copied = rows + r, copied + c
        mlps = 2 * case["layers"] * (2 if case["image_len"] else 1)
        weights = mlps * ((cf + 2) * D * D + 3 * D) * e
        return {"bytes": cols * row * (rows * (cf + 1) + 2 * copied) + weights,
                "flops": cols * rows * 2 * (cf + 2) * D * D}
    if kind == "decode":
        lens = _lens(case)
        per_layer = 2 * case["kv_heads"] * row * (sum(lens) + 2 * len(lens)) + 2 * len(lens) * case["q_heads"] * row
        return {"bytes": case["layers"] * per_layer, "flops": case["layers"] * 4 * case["q_heads"] * D * sum(lens)}
    n = 2 * case["batch"] * case["kv_heads"] * case["seq_len"]                # rows of K and V
    codes = D if case["type"] in ("int8", "fp8") else D // 2
    scale = 0 if case["type"] == "fp8" else e                                 # one for the tensor
    return {"bytes": n * 2 * (row + codes + scale), "flops": n * 4 * D}


def tolerance(case):
    kind = case["kind"]
    if kind in ("press-hook", "press-runner"):
        # rows are moved, not computed; scores that tie within their fp32 sums may be ranked either way, and one such
        # pair moves the rows kept between its two positions by one
        return {"rel": 0.0, "differ": 0.004 if case["window"] else 0.002}
    if kind == "quant":
        return "exact"
    # results are rounded to the storage type: 2^-11 of a value in f16, 2^-8 in bf16; the MLP's hidden activations too
    return {"rel": 1e-3} if case["dtype"] == "f16" else {"rel": 5e-3}
