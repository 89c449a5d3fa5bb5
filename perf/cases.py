"""The work that a user of this package has it do, as cases that can be timed.

A serving program keeps its KV cache packed: it stores a prompt (`prefill`), adds tokens in chunks (`chunk`: chunked
prefill, speculative steps), runs decode steps on the packed cache (`decode`: append of the step's token, then
attention), and gets stretches of cache back as plain tensors (`load`).  A retrieval-like program scores queries
against keys held as codes plus a sign sketch (`estimator`).  A program written for the NumPy classes compresses and
decompresses host arrays (`compressor`: a KV cache, `vectors`: embedding rows).  The listed cases are these seven
paths at the smallest, ordinary and largest sizes they meet; `draw` spreads over the same ranges.

Heads, contexts and formats are those of this repository's benchmark, tests and format policies; values are N(0, 1)
with four channels of every K head scaled by 15, as its benchmark makes them.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import turboquant_plus_amd as tqa

D = 128
DTYPES = {"fp16": torch.float16, "fp32": torch.float32}
# (K, V) formats that the policies name: equal widths, K wider than V, 8-bit K rows, 8-bit rows on both sides
FORMATS = (("turbo3", "turbo3"), ("turbo4", "turbo4"), ("turbo2", "turbo2"), ("turbo4", "turbo3"), ("turbo4", "turbo2"),
           ("q8_0", "turbo3"), ("q8_0", "turbo2"), ("q8_0", "turbo4"), ("q8_0", "q8_0"), ("turbo3", "q8_0"))
HEADS = ((32, 8), (64, 8), (32, 4), (40, 8), (16, 16), (8, 1))     # query heads, KV heads


def listed():
    return [
        # one user's decode step at a short context: launch and host latency are most of it
        dict(name="decode_one_4k", path="decode", k="turbo3", v="turbo3", batch=1, hq=32, hkv=8, head_dim=128, tokens=4000,
             capacity=4096, bias=0, tau=0.0),
        # a full batch at 32K: the benchmark's decode step, the largest one
        dict(name="decode_batch_32k", path="decode", k="turbo3", v="turbo3", batch=16, hq=32, hkv=8, head_dim=128, tokens=32768,
             capacity=32768, bias=0, tau=0.0),
        # long context with 8-bit K rows, 2-bit V rows, a few biased positions per head and the Sparse-V skip
        dict(name="decode_long_q8_turbo2", path="decode", k="q8_0", v="turbo2", batch=4, hq=32, hkv=8, head_dim=128, tokens=131072,
             capacity=131072, bias=64, tau=1e-6),
        # an odd batch of odd length in a cache with room to grow, eight query heads to a KV head
        dict(name="decode_odd_gqa8_turbo4", path="decode", k="turbo4", v="turbo4", batch=6, hq=64, hkv=8, head_dim=128, tokens=10007,
             capacity=16384, bias=0, tau=0.0),
        # the benchmark's store: one layer's K and V of a 32K prompt
        dict(name="prefill_32k_turbo4", path="prefill", k="turbo4", v="turbo4", n_seqs=8, tokens=32768, capacity=32768, dtype="fp16"),
        # a short prompt of one user
        dict(name="prefill_short_turbo3", path="prefill", k="turbo3", v="turbo3", n_seqs=8, tokens=777, capacity=4096, dtype="fp16"),
        # an ordinary prompt in the asymmetric format that the policies start from: 8-bit K rows
        dict(name="prefill_q8_turbo3", path="prefill", k="q8_0", v="turbo3", n_seqs=16, tokens=6001, capacity=8192, dtype="fp16"),
        # the next 512 tokens of a long prompt that is taken in chunks, four users
        dict(name="chunk_512_turbo4", path="chunk", k="turbo4", v="turbo4", n_seqs=32, tokens=512, pos=3584, capacity=8192, dtype="fp16"),
        # a stretch of cache back to fp16 tensors
        dict(name="load_20k_turbo3", path="load", bits_k=3, bits_v=3, n_seqs=8, tokens=20001, dtype="fp16"),
        # keys to codes and sign sketch, then every query against every key: the benchmark's estimator
        dict(name="estimator_64k", path="estimator", bits=3, keys=65536, queries=2048, dtype="fp32", logits="fp32"),
        # the NumPy classes on a KV cache: host arrays in, host arrays out
        dict(name="compressor_2x4x4096", path="compressor", layers=2, heads=4, tokens=4096, d=128, k_bits=3, v_bits=3, dtype="float32"),
        # the NumPy classes on a batch of embedding rows
        dict(name="vectors_256x1536", path="vectors", n=256, d=1536, bits=3, dtype="float32"),
    ]


def _log(rng, lo, hi):
    """An integer from lo to hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("decode", "decode", "decode", "prefill", "prefill", "chunk", "load", "estimator", "compressor", "vectors"))
    if path == "decode":
        k, v = rng.choice(FORMATS)
        hq, hkv = rng.choice(HEADS)
        head_dim = rng.choice((128, 128, 128, 256))
        batch = _log(rng, 1, 32)
        tokens = _log(rng, 256, min(131072, 16 * 32768 * 8 * 128 // (batch * hkv * head_dim)))
        capacity = tokens if rng.random() < 0.5 else -(-tokens // 4096) * 4096
        return dict(path=path, k=k, v=v, batch=batch, hq=hq, hkv=hkv, head_dim=head_dim, tokens=tokens, capacity=capacity,
                    bias=rng.choice((0, 0, 0, 64)), tau=rng.choice((0.0, 0.0, 0.0, 1e-6)))
    if path == "prefill":
        k, v = rng.choice(FORMATS)
        n_seqs = rng.choice((4, 8, 16, 40, 64))
        tokens = _log(rng, 32, 262144 // n_seqs)
        return dict(path=path, k=k, v=v, n_seqs=n_seqs, tokens=tokens, capacity=-(-tokens // 2048) * 2048,
                    dtype=rng.choice(("fp16", "fp16", "fp32")))
    if path == "chunk":
        k, v = rng.choice(FORMATS)
        n_seqs, tokens, pos = rng.choice((8, 16, 32, 64)), _log(rng, 2, 2048), rng.choice((0, 1, 1)) * _log(rng, 1, 14000)
        return dict(path=path, k=k, v=v, n_seqs=n_seqs, tokens=tokens, pos=pos, capacity=16384,
                    dtype=rng.choice(("fp16", "fp16", "fp32")))
    if path == "load":
        n_seqs = rng.choice((1, 8, 16, 64))
        return dict(path=path, bits_k=rng.choice((2, 3, 4)), bits_v=rng.choice((2, 3, 4)), n_seqs=n_seqs,
                    tokens=_log(rng, 64, 262144 // n_seqs), dtype=rng.choice(("fp16", "fp16", "fp32")))
    if path == "estimator":
        return dict(path=path, bits=rng.choice((2, 3, 4)), keys=_log(rng, 500, 65536), queries=_log(rng, 1, 2048),
                    dtype=rng.choice(("fp16", "fp32")), logits=rng.choice(("fp16", "fp32")))
    if path == "compressor":
        layers, heads = rng.choice(((1, 4), (2, 4), (1, 8), (2, 2), (4, 2)))
        d = rng.choice((64, 96, 128, 256))
        return dict(path=path, layers=layers, heads=heads, tokens=_log(rng, 16, 8 * 4096 * 128 // (layers * heads * d)), d=d,
                    k_bits=rng.choice((2, 3, 4)), v_bits=rng.choice((2, 3, 4)), dtype=rng.choice(("float32", "float64")))
    d = rng.choice((384, 768, 1024, 1536))
    return dict(path=path, n=_log(rng, 1, 256 * 1536 // d), d=d, bits=rng.choice((2, 3, 4)), dtype=rng.choice(("float32", "float64")))


# ---- what a program keeps: one quantiser per format for all its layers, steps and inputs --------------------------------

@functools.lru_cache(maxsize=None)
def _layer(k, v):
    return tqa.LayerKV(tqa.LayerFormat(k, v))


@functools.lru_cache(maxsize=None)
def _codec(bits, seed, projection=None):
    return tqa.TurboCodec(bits, seed=seed, projection=projection, projection_seed=2 if projection else None)


@functools.lru_cache(maxsize=None)
def _compressor(d, k_bits, v_bits):
    return tqa.KVCacheCompressor(d, k_bits=k_bits, v_bits=v_bits)


@functools.lru_cache(maxsize=4)
def _quantizer(d, bits):
    return tqa.TurboQuant(d, bits)


def _rows(gen, n_seqs, tokens, dtype=torch.float16, outliers=0):
    """N(0, 1) rows [n_seqs, tokens, 128] on the GPU; `outliers` channels of every sequence scaled by 15."""
    x = torch.randn((n_seqs, tokens, D), generator=gen, device="cuda", dtype=torch.float32)
    if outliers:
        ch = torch.argsort(torch.rand((n_seqs, D), generator=gen, device="cuda"), dim=-1)[:, :outliers]
        x *= torch.ones((n_seqs, D), device="cuda").scatter_(1, ch, 15.0)[:, None]
    return x.to(dtype)


def _filled_cache(layer, gen, n_seqs, rows, capacity):
    """Packed caches for `capacity` rows per sequence with the first `rows` of them written, a few sequences at a time
    (every sequence's part of a cache is a cache of its own)."""
    kc, vc = layer.new_cache(n_seqs, capacity)
    if rows:
        per_k, per_v = kc.numel() // n_seqs, vc.numel() // n_seqs
        step = max(1, min(n_seqs, (1 << 18) // rows))
        for s in range(0, n_seqs, step):
            e = min(n_seqs, s + step)
            layer.prefill(_rows(gen, e - s, rows, outliers=4), _rows(gen, e - s, rows), kc[s * per_k:e * per_k],
                          vc[s * per_v:e * per_v], capacity)
    return kc, vc


def _host_rows(seed, shape, dtype):
    return np.random.default_rng(seed).standard_normal(shape, dtype=np.float32).astype(dtype)


def prepare(case, seed):
    path = case["path"]
    if path == "compressor":
        c = _compressor(case["d"], case["k_bits"], case["v_bits"])
        shape = (case["layers"], case["heads"], case["tokens"], case["d"])
        return dict(path=path, c=c, k=_host_rows(2 * seed, shape, case["dtype"]), v=_host_rows(2 * seed + 1, shape, case["dtype"]))
    if path == "vectors":
        return dict(path=path, q=_quantizer(case["d"], case["bits"]), x=_host_rows(seed, (case["n"], case["d"]), case["dtype"]))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if path == "estimator":
        # the sketch's projection is a Gaussian matrix drawn from seed 2, as the benchmark has it
        return dict(path=path, codec=_codec(case["bits"], 42, "gaussian"),
                    keys=_rows(gen, 1, case["keys"], DTYPES[case["dtype"]])[0], q=_rows(gen, 1, case["queries"])[0],
                    n=case["keys"], logits=DTYPES[case["logits"]])
    if path == "load":
        kc, vc = _codec(case["bits_k"], 42), _codec(case["bits_v"], 542)
        n, t = case["n_seqs"], case["tokens"]
        return dict(path=path, kc=kc, vc=vc, kp=kc.store(_rows(gen, n, t, outliers=4), kind="k"), vp=vc.store(_rows(gen, n, t), kind="v"),
                    n=n, tokens=t, dtype=DTYPES[case["dtype"]])
    layer = _layer(case["k"], case["v"])
    if path == "decode":
        two = case["head_dim"] // D          # rows of a token: a head of 256 dims is two of 128
        n_seqs, t, cap = case["batch"] * case["hkv"], case["tokens"], case["capacity"]
        kc, vc = _filled_cache(layer, gen, n_seqs, two * (t - 1), two * cap)
        attn = layer.attention(case["batch"], case["hq"], case["hkv"], t, capacity=cap, sparse_v_tau=case["tau"], head_dim=case["head_dim"])
        q = _rows(gen, case["batch"] * case["hq"], two).reshape(case["batch"], case["hq"], case["head_dim"])
        sb = None
        if case["bias"]:   # +6 on that many positions of every head
            shape = (case["batch"], case["hq"], case["bias"])
            edge = torch.arange(case["bias"] + 1, device="cuda", dtype=torch.float64) * (t / case["bias"])
            lo, hi = edge[:-1].floor().to(torch.int64), edge[1:].floor().to(torch.int64)
            pos = (lo + (torch.rand(shape, generator=gen, device="cuda") * (hi - lo)).to(torch.int64)).to(torch.int32)
            sb = (pos, torch.full(shape, 6.0, device="cuda"))
        return dict(path=path, layer=layer, attn=attn, kc=kc, vc=vc, k=_rows(gen, n_seqs, two, outliers=4), v=_rows(gen, n_seqs, two), q=q,
                    sb=sb, pos=two * (t - 1), capacity=two * cap)
    n, t, dt = case["n_seqs"], case["tokens"], DTYPES[case["dtype"]]
    pos = case.get("pos", 0)
    kc, vc = _filled_cache(layer, gen, n, pos, case["capacity"])
    return dict(path=path, layer=layer, k=_rows(gen, n, t, dt, outliers=4), v=_rows(gen, n, t, dt), kc=kc, vc=vc, pos=pos,
                capacity=case["capacity"])


def run(s):
    path = s["path"]
    if path == "decode":
        s["layer"].append(s["k"], s["v"], s["kc"], s["vc"], s["pos"], s["capacity"])
        return s["attn"](s["q"], s["kc"], s["vc"], sparse_bias=s["sb"]), s["kc"], s["vc"]
    if path == "prefill":
        return s["layer"].prefill(s["k"], s["v"], s["kc"], s["vc"], s["capacity"])
    if path == "chunk":
        return s["layer"].append(s["k"], s["v"], s["kc"], s["vc"], s["pos"], s["capacity"])
    if path == "load":
        if s["dtype"] == torch.float16:
            return s["kc"].load_kv(s["vc"], s["kp"], s["vp"], s["n"], s["tokens"])
        return (s["kc"].load(s["kp"], s["n"], s["tokens"], kind="k", dtype=s["dtype"]),
                s["vc"].load(s["vp"], s["n"], s["tokens"], kind="v", dtype=s["dtype"]))
    if path == "estimator":
        packed, bits, norms = s["codec"].store_qjl(s["keys"])
        return packed, bits, norms, s["codec"].score_tile(s["q"], packed, bits, norms, s["n"], out_dtype=s["logits"])
    if path == "compressor":
        c = s["c"].compress(s["k"], s["v"])
        k, v = s["c"].decompress(c)
        return (k, v, [[(x.mse_indices, x.vector_norms, x.qjl_signs, x.residual_norms) for x in row] for row in c.k_compressed],
                c.v_indices, c.v_norms)
    c = s["q"].quantize(s["x"])
    return c.mse_indices, c.vector_norms, c.qjl_signs, c.residual_norms, s["q"].dequantize(c)


def _row_bytes(fmt):
    return 136 if fmt == "q8_0" else 16 * int(fmt[-1]) + 2


def work(case):
    path = case["path"]
    rotate = 7 * D + 12 * D      # butterfly, norm and quantiser (or look-up) of one row
    if path == "decode":
        two = case["head_dim"] // D
        rows = case["batch"] * case["hkv"] * case["tokens"] * two
        new = case["batch"] * case["hkv"] * two
        io = case["batch"] * case["hq"] * (case["head_dim"] * (2 + 4) + 8 * case["bias"])
        return {"bytes": (rows + new) * (_row_bytes(case["k"]) + _row_bytes(case["v"])) + 2 * new * 2 * D + io,
                "flops": 4 * case["batch"] * case["hq"] * case["tokens"] * case["head_dim"]}
    if path in ("prefill", "chunk"):
        n, size = case["n_seqs"] * case["tokens"], 2 if case["dtype"] == "fp16" else 4
        return {"bytes": n * (2 * D * size + _row_bytes(case["k"]) + _row_bytes(case["v"])), "flops": 2 * n * rotate}
    if path == "load":
        n, size = case["n_seqs"] * case["tokens"], 2 if case["dtype"] == "fp16" else 4
        return {"bytes": n * (2 * D * size + 16 * (case["bits_k"] + case["bits_v"]) + 4), "flops": 2 * n * rotate}
    if path == "estimator":
        size = {"fp16": 2, "fp32": 4}
        keys = case["keys"] * (D * size[case["dtype"]] + 2 * (16 * case["bits"] + 2 + 16 + 2))    # written, then read by the scores
        return {"bytes": keys + case["queries"] * (2 * D + case["keys"] * size[case["logits"]]),
                "flops": case["keys"] * (2 * D * D + rotate) + 2 * case["queries"] * case["keys"] * 2 * D}
    size = 4 if case["dtype"] == "float32" else 8
    if path == "compressor":
        n, d = case["layers"] * case["heads"] * case["tokens"], case["d"]
        # K: rotate, reconstruct, project; V: rotate; back: three products
        return {"bytes": n * (2 * d * (size + 8 + 8) + d + 24) + n * (2 * 8 * d + d + 24), "flops": 7 * 2 * n * d * d}
    n, d = case["n"], case["d"]
    return {"bytes": n * (d * (size + 8 + 1 + 8) + 16) + n * (9 * d + 16), "flops": 5 * 2 * n * d * d}


def tolerance(case):
    """About four times what the paths measure against the same arithmetic in 64 bits on the stored codes (attention and
    scores: fp16 operands; fp16 loads: fp16 centroids; packed bytes: codes whose rotated value lies on a decision boundary
    to within 32-bit rounding, and norms next to a rounding midpoint of fp16).  8-bit rows and the NumPy classes'
    indices and signs are whole numbers that have one right value."""
    path = case["path"]
    if path == "decode":
        return {"rel": 3e-3, "max": 2.5e-2, "differ": 4e-5}
    if path in ("prefill", "chunk"):
        return "exact" if case["k"] == case["v"] == "q8_0" else {"differ": 4e-5}
    if path == "load":
        return {"rel": 1.5e-3, "max": 1.4e-2} if case["dtype"] == "fp16" else {"rel": 1e-6}
    if path == "estimator":
        return {"rel": 1.8e-3, "max": 1.2e-2, "differ": 4e-5}
    return {"rel": 1e-12, "max": 1e-10}
