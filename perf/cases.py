"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values. Its "kind" names the call:

- generate   one short request on one layer, called step by step as an eager decode loop does: a new cache, the
             prompt's update, then one-token updates with their attention;
- decode     one token's attention over filled compressed caches, one call per layer (`graph`: the layers' calls are
             captured once and replayed, as a serving loop does; else they are called);
- ragged     one decode step of a batch of sequences of different lengths (append, drain, attention);
- dense      one token's attention over the uncompressed caches of outlier / skipped layers;
- store      a prompt's keys and values into a new compressed cache (the fused prefill path keeps only the codes);
- fetch      the same through update_and_fetch, which returns the dense float32 keys and values;
- prefill    causal attention of a chunk of query tokens over the packed codes;
- quantizer  TurboQuantMSE / TurboQuantProd: quantize and dequantize a set of vectors.

Keys are N(0, 1) times a per-channel LogNormal(0, 0.5) factor (key channels differ in scale in trained models), values
N(0, 1), queries N(0, 1) times 2 (scores then spread over several units, as attention scores do).
A vector with a rotated coordinate within float32 rounding of a cell boundary (or a sketch projection that close to
zero) has two right codes, and one other code moves an attention output by far more than its arithmetic does: such
vectors, about 1 in 300 (1 in 50 with a sketch), are replaced by the one before them.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("mlx-turboquant_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from turboquant_amd import TurboQuantKVCache, TurboQuantMSE, TurboQuantProd  # noqa: E402
from turboquant_amd.patch import FP16KVCache  # noqa: E402
from turboquant_amd.ragged import RaggedKVBatch  # noqa: E402

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
WINDOW = 128  # the cache's default residual window


def listed():
    return [
        # the smallest request: a 400-token prompt on a small grouped-query layer, 16 tokens generated eagerly
        dict(name="generate_short", kind="generate", dtype="fp16", d=128, hkv=2, hq=8, batch=1, prompt=400, steps=16,
             kbits=4, vbits=2, sink=16, window=64, qjl=0),
        # one attention call over a short chat context, eager: latency only
        dict(name="decode_1k_eager", kind="decode", graph=False, layers=1, dtype="fp16", d=128, hkv=8, hq=32, batch=1,
             tokens=1000, kbits=4, vbits=2, sink=0, qjl=0),
        # the benchmark's decode step: 32 layers of an 8B-class model over a 32K context
        dict(name="decode_32k", kind="decode", graph=True, layers=32, dtype="fp16", d=128, hkv=8, hq=32, batch=1,
             tokens=32768, kbits=4, vbits=2, sink=128, qjl=0),
        # symmetric 4-bit caches of a bf16 model whose query-head ratio is 7 (28 heads on 4)
        dict(name="decode_bf16_gqa7", kind="decode", graph=True, layers=16, dtype="bf16", d=128, hkv=4, hq=28, batch=1,
             tokens=16001, kbits=4, vbits=4, sink=0, qjl=0),
        # head_dim 64 (1B-class models), a batch of two mid-length contexts
        dict(name="decode_d64", kind="decode", graph=True, layers=16, dtype="bf16", d=64, hkv=8, hq=32, batch=2,
             tokens=8229, kbits=4, vbits=2, sink=4, qjl=0),
        # head_dim 256 with few kv heads, at the widths few kv heads are upgraded to
        dict(name="decode_d256", kind="decode", graph=True, layers=16, dtype="bf16", d=256, hkv=2, hq=8, batch=1,
             tokens=12000, kbits=4, vbits=3, sink=0, qjl=0),
        # continuous batching: 16 sequences of 4K-32K tokens with the QJL sketch
        dict(name="ragged_qjl", kind="ragged", batch=16, hkv=8, hq=32, d=128, lo=4096, hi=32000, kbits=4, vbits=2,
             sink=0, window=128, qjl=128),
        # an outlier model's uncompressed layers over a 64K context
        dict(name="dense_64k", kind="dense", graph=True, layers=6, dtype="fp16", d=128, hkv=8, hq=32, batch=1,
             tokens=65536),
        # a 128K prompt into the cache, drained in 4096-token chunks
        dict(name="store_128k", kind="store", dtype="fp16", d=128, hkv=8, batch=1, tokens=131072, kbits=3, vbits=2,
             sink=0, chunk=4096, qjl=0),
        # the dense-contract prefill of a bf16 model (update_and_fetch feeding the model's own attention)
        dict(name="fetch_bf16_8k", kind="fetch", dtype="bf16", d=128, hkv=8, batch=1, tokens=8192, kbits=4, vbits=2,
             sink=0, chunk=0, qjl=0),
        # a 1,024-token prompt chunk attending over a 32K context
        dict(name="prefill_32k", kind="prefill", dtype="fp16", d=128, hkv=8, hq=32, batch=1, tokens=32768, nq=1024,
             kbits=4, vbits=2, sink=128, qjl=0),
        # vectors through the two-stage quantizer (retrieval / offline use)
        dict(name="prod_64k", kind="quantizer", prod=True, dtype="fp32", d=128, bits=4, n=65536),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["generate", "decode", "decode", "decode", "decode", "ragged", "dense", "store", "fetch",
                       "prefill", "quantizer"])
    dtype = rng.choice(["fp16", "bf16"])
    hkv = rng.choice([1, 2, 4, 8])
    hq = hkv * rng.choice([1, 2, 4, 4, 5, 7, 8])
    kbits, vbits = rng.choice([(4, 2), (4, 2), (4, 4), (3, 2), (4, 3), (3, 3), (3.5, 3.5), (3.5, 2)])
    d = rng.choice([128, 128, 128, 64, 64, 96, 256])
    sink = rng.choice([0, 0, 4, 128])
    qjl = rng.choice([0, 0, 0, 0, 0, 32])
    if kind == "generate":
        return dict(kind=kind, dtype=dtype, d=d, hkv=hkv, hq=hq, batch=rng.choice([1, 1, 2]),
                    prompt=_log(rng, 40, 2000), steps=rng.randint(4, 16), kbits=kbits, vbits=vbits, sink=sink,
                    window=rng.choice([32, 64, 128]), qjl=qjl)
    if kind == "decode":
        batch, tokens = rng.choice([1, 1, 2, 4]), _log(rng, 400, 32768)
        if tokens < 2000:
            return dict(kind=kind, graph=False, layers=1, dtype=dtype, d=d, hkv=hkv, hq=hq, batch=batch, tokens=tokens,
                        kbits=kbits, vbits=vbits, sink=sink, qjl=qjl)
        return dict(kind=kind, graph=True, layers=8, dtype=dtype, d=d, hkv=hkv, hq=hq, batch=batch,
                    tokens=min(tokens, 49152 // batch), kbits=kbits, vbits=vbits, sink=sink, qjl=qjl)
    if kind == "ragged":
        lo = _log(rng, 300, 4096)
        kb, vb = rng.choice([(4, 2), (4, 2), (3, 2), (4, 4)])
        return dict(kind=kind, batch=rng.randint(2, 16), hkv=hkv, hq=hkv * rng.choice([1, 2, 4, 8]), d=128, lo=lo,
                    hi=lo * rng.randint(2, 7), kbits=kb, vbits=vb, sink=rng.choice([0, 128]), window=128,
                    qjl=rng.choice([0, 128]) if (kb, vb) == (4, 2) else 0)
    if kind == "dense":
        return dict(kind=kind, graph=True, layers=6, dtype=dtype, d=128, hkv=hkv, hq=hkv * rng.choice([1, 2, 4, 8]),
                    batch=1, tokens=_log(rng, 1000, 65536))
    if kind == "store":
        return dict(kind=kind, dtype=dtype, d=d, hkv=hkv, batch=rng.choice([1, 2]), tokens=_log(rng, 400, 32768),
                    kbits=kbits, vbits=vbits, sink=sink, chunk=rng.choice([0, 256]), qjl=qjl)
    if kind == "fetch":
        return dict(kind=kind, dtype=dtype, d=d, hkv=hkv, batch=1, tokens=_log(rng, 400, 16384), kbits=kbits,
                    vbits=vbits, sink=sink, chunk=0, qjl=qjl)
    if kind == "prefill":
        kb, vb = rng.choice([(4, 2), (4, 4), (3, 2), (3, 3)])
        nq = _log(rng, 16, 512)
        return dict(kind=kind, dtype=dtype, d=128, hkv=hkv, hq=hq, batch=1, tokens=nq + _log(rng, 300, 16384), nq=nq,
                    kbits=kb, vbits=vb, sink=sink, qjl=0)
    prod = rng.choice([True, False])
    return dict(kind="quantizer", prod=prod, dtype=rng.choice(["fp32", "fp16", "bf16"]), d=d,
                bits=rng.choice([2, 3, 4]), n=_log(rng, 64, 65536))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _kv(case, g, batch, tokens):
    """Keys and values (batch, hkv, tokens, d)."""
    hkv, d, dtype = case["hkv"], case["d"], DTYPES[case.get("dtype", "fp16")]
    sc = torch.exp(0.5 * torch.randn(hkv, 1, d, device=DEV, generator=g))
    k = (torch.randn(batch, hkv, tokens, d, device=DEV, generator=g) * sc).to(dtype)
    v = torch.randn(batch, hkv, tokens, d, device=DEV, generator=g).to(dtype)
    if case["kind"] == "dense":
        return k, v
    return _untied(k, case["kbits"], case["qjl"]), _untied(v, case["vbits"], case["qjl"])


def _untied(x, bits, m):
    """x (..., T, d) with every vector that has two right codes replaced by the nearest one before it that has not (at
    the start of a row: by the row's first)."""
    d = x.shape[-1]
    rot, books, split, proj = _const(d, bits, m)
    rows = x.reshape(-1, x.shape[-2], d)
    step = max(1, (1 << 18) // rows.shape[1])
    pos = torch.arange(rows.shape[1], device=x.device)
    out = []
    for part in rows.split(step):
        f = part.double()
        n = f.square().sum(-1, keepdim=True).sqrt().clamp_min(1e-10)
        y = (f / n) @ rot.T
        tied = torch.zeros(part.shape[:-1], dtype=torch.bool, device=x.device)
        for z, (_, bnd) in zip((y[..., :split], y[..., split:]), books):
            if z.shape[-1]:
                z = z.contiguous()
                above = torch.bucketize(z, bnd)
                gap = torch.minimum((z - bnd[(above - 1).clamp_min(0)]).abs(),
                                    (z - bnd[above.clamp_max(len(bnd) - 1)]).abs())
                tied |= (gap < 2e-7).any(-1)
        if m:
            res = f - _exact_codec(part, bits, 0)[1]
            tied |= ((res @ proj.T).abs() < 1e-5 * n).any(-1)
        src = torch.where(tied, -1, pos).cummax(-1).values
        src = torch.where(src < 0, (~tied).to(torch.int8).argmax(-1, keepdim=True), src)
        out.append(part.gather(1, src[..., None].expand(-1, -1, d)))
    return torch.cat(out).reshape(x.shape)


def _q(g, batch, hq, nq, d, dtype):
    return (2 * torch.randn(batch, hq, nq, d, device=DEV, generator=g)).to(DTYPES[dtype])


def _cache(case):
    return TurboQuantKVCache(head_dim=case["d"], num_kv_heads=case["hkv"], key_bits=case["kbits"],
                             value_bits=case["vbits"], residual_window=case.get("window", WINDOW),
                             fp16_sink_size=case["sink"], chunk_size=case.get("chunk", 0),
                             qjl_correction=case.get("qjl", 0) > 0, qjl_n_proj=case.get("qjl", 0) or 32)


def _lengths(case):
    """The ragged batch's sequence lengths, spread over [lo, hi]."""
    return [case["lo"] + int((case["hi"] - case["lo"]) * ((0.5 + 0.6180339887 * i) % 1.0))
            for i in range(case["batch"])]


def _generate_inputs(case, seed):
    g = _gen(seed)
    k, v = _kv(case, g, case["batch"], case["prompt"] + case["steps"])
    q = [_q(g, case["batch"], case["hq"], 1, case["d"], case["dtype"]) for _ in range(case["steps"])]
    return k, v, q


def _layer_inputs(case, g):
    k, v = _kv(case, g, case["batch"], case["tokens"])
    return k, v, _q(g, case["batch"], case["hq"], case.get("nq", 1), case["d"], case["dtype"])


def _ragged_inputs(case, seed):
    """Per sequence (K, V) (hkv, T, d), then the step's token and query."""
    g = _gen(seed)
    seqs = [tuple(x[0] for x in _kv(case, g, 1, t)) for t in _lengths(case)]
    k, v = _kv(case, g, 1, case["batch"])  # the batch along the token axis: one token for each sequence
    return seqs, k[0].transpose(0, 1).contiguous(), v[0].transpose(0, 1).contiguous(), \
        _q(g, case["batch"], case["hq"], 1, case["d"], "fp16")[:, :, 0].contiguous()


def _vectors(case, seed):
    x = torch.randn(case["n"], case["d"], device=DEV, generator=_gen(seed)).to(DTYPES[case["dtype"]])
    return _untied(x[None], case["bits"] - 1 if case["prod"] else case["bits"], case["d"] if case["prod"] else 0)[0]


# --------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "generate":
        k, v, q = _generate_inputs(case, seed)
        p = case["prompt"]
        cut = lambda x: [x[:, :, :p].contiguous()] + [x[:, :, i:i + 1].contiguous() for i in range(p, x.shape[2])]  # noqa: E731
        return {"case": case, "k": cut(k), "v": cut(v), "q": q}
    if kind in ("decode", "dense"):
        g = _gen(seed)
        caches, qs = [], []
        for _ in range(case["layers"]):
            k, v, q = _layer_inputs(case, g)
            c = FP16KVCache() if kind == "dense" else _cache(case)
            c.update(k, v)
            caches.append(c)
            qs.append(q)
        s = {"case": case, "caches": caches, "q": qs}
        if case["graph"]:
            s["out"] = [torch.empty(q.shape, dtype=torch.float32, device=DEV) for q in qs]
            calls = lambda: [c.attend(q, out=o) for c, q, o in zip(caches, qs, s["out"])]  # noqa: E731
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                calls()
            torch.cuda.current_stream().wait_stream(stream)
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"], stream=stream):
                calls()
        return s
    if kind == "ragged":
        seqs, k, v, q = _ragged_inputs(case, seed)
        b = RaggedKVBatch(case["batch"], case["hkv"], head_dim=case["d"], key_bits=case["kbits"],
                          value_bits=case["vbits"], residual_window=case["window"], fp16_sink_size=case["sink"],
                          qjl_n_proj=case["qjl"])
        for i, (sk, sv) in enumerate(seqs):
            b.load(i, sk, sv)
        return {"case": case, "batch": b, "k": k, "v": v, "q": q}
    if kind in ("store", "fetch"):
        k, v = _kv(case, _gen(seed), case["batch"], case["tokens"])
        return {"case": case, "k": k, "v": v}
    if kind == "prefill":
        k, v, q = _layer_inputs(case, _gen(seed))
        c = _cache(case)
        c.update(k, v)
        return {"case": case, "cache": c, "q": q}
    return {"case": case, "x": _vectors(case, seed),
            "quantizer": (TurboQuantProd if case["prod"] else TurboQuantMSE)(case["d"], bits=case["bits"])}


# ------------------------------------------------------------------- run
def _state(cache):
    """What an update leaves in the cache: the packed codes, norms and sketch of both sides."""
    out = []
    for side in ("k", "v"):
        out += [t for t in cache.packed(side) if t is not None]
        sk = cache.sketch(side)
        if sk is not None:
            out += list(sk)
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "generate":
        c = _cache(case)
        c.update(state["k"][0], state["v"][0])
        outs = []
        for k, v, q in zip(state["k"][1:], state["v"][1:], state["q"]):
            c.update(k, v)
            outs.append(c.attend(q))
        return {"out": outs, "state": _state(c)}
    if kind in ("decode", "dense"):
        if case["graph"]:
            state["graph"].replay()
            return state["out"]
        return [c.attend(q) for c, q in zip(state["caches"], state["q"])]
    if kind == "ragged":
        b = state["batch"]
        b.step(state["k"], state["v"])
        out = b.attend(state["q"])
        n = int(b.comp_len.min())  # every sequence's codes up to the shortest's length, its drained token among them
        s = [out, b.ring_k, b.ring_v]
        for st in (b.kstore, b.vstore):
            s += [t[:, :, :n] for t in (st.codes_hi, st.norms, st.signs, st.gamma) if t is not None and n]
        return s
    if kind == "store":
        c = _cache(case)
        c.update(state["k"], state["v"])
        return _state(c) + [t for t in (c.keys, c.values) if t is not None]
    if kind == "fetch":
        return _cache(case).update_and_fetch(state["k"], state["v"])
    if kind == "prefill":
        return state["cache"].attend(state["q"])
    qt = state["quantizer"].quantize(state["x"])
    out = [qt.packed_indices, qt.norms, state["quantizer"].dequantize(qt)]
    return out + [qt.qjl_signs, qt.qjl_norms] if case["prod"] else out


# ------------------------------------------------------------------ work
def _row_bytes(d, bits, m):
    """Bytes of one packed vector: codes, float32 norm, and the sketch's signs and residual norm."""
    hi, lo, split = _split(bits, d)
    return (split * hi + (d - split) * lo) // 8 + 4 + (((m + 31) // 32) * 4 + 4 if m else 0)


def _split(bits, d):
    return (int(bits) + 1, int(bits), d // 2) if bits != int(bits) else (int(bits), int(bits), d)


def _compressed(case, total):
    """(sink, compressed, residual) lengths after one update of ``total`` tokens into a new cache."""
    s = min(case["sink"], total)
    n, w, chunk = total - s, case.get("window", WINDOW), case.get("chunk", 0)
    if chunk <= 0:
        c = n - w if n > 2 * w else 0
    else:
        c = (n - w) // chunk * chunk if n >= w + chunk else 0
    return s, c, n - c


def _attend_work(d, hkv, hq, nq, lens, case, q_bytes, kv_bytes):
    """Bytes and operations of attention over sequences of (sink, compressed, residual) ``lens``; the causal queries
    see the tokens up to their own."""
    row = _row_bytes(d, case["kbits"], case.get("qjl", 0)) + _row_bytes(d, case["vbits"], case.get("qjl", 0))
    by = fl = 0
    for s, c, r in lens:
        by += hkv * (c * row + (s + r) * 2 * d * kv_bytes) + hq * nq * d * (q_bytes + 4)
        fl += 4 * hq * d * (nq * (s + c + r) - nq * (nq - 1) // 2)
    return {"bytes": by, "flops": fl}


def work(case):
    kind, d = case["kind"], case["d"]
    es = {"fp16": 2, "bf16": 2, "fp32": 4}[case.get("dtype", "fp16")]
    if kind == "generate":
        n = case["batch"] * case["hkv"]
        total = {"bytes": 2 * n * (case["prompt"] + case["steps"]) * d * es, "flops": 0}
        comp, res, sink = 0, 0, 0
        for t in [case["prompt"]] + [1] * case["steps"]:
            a = min(case["sink"] - sink, t)
            sink, res = sink + a, res + t - a
            if res > 2 * case["window"]:
                moved, res = res - case["window"], case["window"]
                comp += moved
                total["bytes"] += n * moved * (_row_bytes(d, case["kbits"], case["qjl"])
                                               + _row_bytes(d, case["vbits"], case["qjl"]))
                total["flops"] += n * moved * 2 * (2 * d * d + 2 * d * case["qjl"])
            if sink + res + comp > case["prompt"]:
                w = _attend_work(d, case["hkv"], case["hq"], 1, [(sink, comp, res)] * case["batch"], case, es, es)
                total = {x: total[x] + w[x] for x in total}
        return total
    if kind == "decode":
        w = _attend_work(d, case["hkv"], case["hq"], 1, [_compressed(case, case["tokens"])] * case["batch"], case, es,
                         es)
        return {x: w[x] * case["layers"] for x in w}
    if kind == "dense":
        t = case["tokens"] * case["batch"] * case["layers"]
        return {"bytes": t * case["hkv"] * 2 * d * es + case["layers"] * case["batch"] * case["hq"] * d * (es + 4),
                "flops": 4 * t * case["hq"] * d}
    if kind == "ragged":
        lens = []
        for t in _lengths(case):
            s, w = min(t, case["sink"]), case["window"]
            r = min(t + 1 - s, w)
            lens.append((s, t + 1 - s - r, r))
        return _attend_work(d, case["hkv"], case["hq"], 1, lens, case, 2, 2)
    if kind == "prefill":
        return _attend_work(d, case["hkv"], case["hq"], case["nq"], [_compressed(case, case["tokens"])] * case["batch"],
                            case, es, es)
    if kind == "quantizer":
        bits, m = (case["bits"] - 1, d) if case["prod"] else (case["bits"], 0)
        return {"bytes": case["n"] * (d * es + 2 * _row_bytes(d, bits, m) + d * 4),
                "flops": case["n"] * 2 * (2 * d * d + 2 * d * m)}
    n = case["batch"] * case["hkv"]
    _, c, _ = _compressed(case, case["tokens"])
    m = case["qjl"]
    row = _row_bytes(d, case["kbits"], m) + _row_bytes(d, case["vbits"], m)
    if kind == "store":
        return {"bytes": n * (2 * case["tokens"] * d * es + c * row + 2 * (case["tokens"] - c) * d * es),
                "flops": n * c * 2 * (2 * d * d + 2 * d * m)}
    return {"bytes": n * (2 * case["tokens"] * d * (es + (4 if c else 0)) + c * row),
            "flops": n * c * 2 * (4 * d * d + 4 * d * m)}


# ------------------------------------------------------------- tolerance
def tolerance(case):
    """Float outputs are 32-bit sums throughout; prefill rounds its softmax weights to fp16 (2e-4 against 64 bits).
    Packed bytes: no input vector has a coordinate near a cell boundary."""
    if case["kind"] == "prefill":
        return {"rel": 1e-3, "max": 2e-2}
    return {"rel": 1e-5, "max": 1e-3, "differ": 2e-6}


# ----------------------------------------------------------------- exact
_consts = {}


def _const(d, bits, m):
    """(R, [(centroids, boundaries) of dims [0, split) and [split, d)], split, S) in float64 on the GPU: the seeded
    rotation and projection, and the shipped codebooks of this width."""
    key = (d, bits, m)
    if key not in _consts:
        g = np.random.RandomState(42).randn(d, d).astype(np.float32)
        q, r = np.linalg.qr(g)
        sg = np.sign(np.diag(r))
        sg[sg == 0] = 1
        rot = (q * sg[None, :]).astype(np.float32)
        hi, lo, split = _split(bits, d)
        books = []
        for b in (hi, lo):
            with np.load(os.path.join(_PKG, "turboquant_amd", "codebooks", f"codebook_d{d}_b{b}.npz")) as z:
                books.append(tuple(torch.from_numpy(z[n].astype(np.float64)).to(DEV)
                                   for n in ("centroids", "boundaries")))
        s = np.random.RandomState(12345).randn(m, d).astype(np.float32) if m else None
        _consts[key] = (torch.from_numpy(rot.astype(np.float64)).to(DEV), books, split,
                        None if s is None else torch.from_numpy(s.astype(np.float64)).to(DEV))
    return _consts[key]


def _exact_codec(x, bits, m):
    """(norms, x dequantized with the sketch's correction, x dequantized, sketch signs, residual norms) of vectors x
    (..., d), in float64."""
    d = x.shape[-1]
    rot, books, split, proj = _const(d, bits, m)
    x = x.double()
    n = x.square().sum(-1, keepdim=True).sqrt()
    y = (x / n.clamp_min(1e-10)) @ rot.T
    c = torch.cat([cen[torch.bucketize(part.contiguous(), bnd, right=False)]
                   for part, (cen, bnd) in zip((y[..., :split], y[..., split:]), books) if part.shape[-1]], dim=-1)
    plain = n * (c @ rot)
    if not m:
        return n[..., 0], plain, plain, None, None
    res = x - plain
    signs = res @ proj.T >= 0
    gamma = res.square().sum(-1, keepdim=True).sqrt()
    corr = plain + math.sqrt(math.pi / 2) / d * gamma * (torch.where(signs, 1.0, -1.0).double() @ proj)
    return n[..., 0], corr, plain, signs, gamma[..., 0]


def _exact_tokens(k, v, case, sink, comp):
    """Keys and values as the cache holds them: tokens [sink, sink + comp) compressed (batch, hkv, T, d)."""
    out = []
    for x, bits in ((k, case["kbits"]), (v, case["vbits"])):
        y = x.double()
        if comp:
            y = y.clone()
            y[:, :, sink:sink + comp] = _exact_codec(x[:, :, sink:sink + comp], bits, case.get("qjl", 0))[1]
        out.append(y)
    return out


def _exact_attend(q, k, v):
    """softmax(q k^T / sqrt(d)) v, the queries the last tokens of the context: q (batch, hq, nq, d)."""
    B, hq, nq, d = q.shape
    g, t = hq // k.shape[1], k.shape[2]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for b in range(B):
        for h in range(k.shape[1]):
            s = (q[b, h * g:(h + 1) * g].double().reshape(-1, d) @ k[b, h].T.contiguous()) * d ** -0.5
            if nq > 1:
                s = s.reshape(g, nq, t)
                s.masked_fill_(torch.arange(t, device=DEV)[None, :] > torch.arange(nq, device=DEV)[:, None] + t - nq,
                               float("-inf"))
                s = s.reshape(-1, t)
            out[b, h * g:(h + 1) * g] = (torch.softmax(s, dim=-1) @ v[b, h]).reshape(g, nq, d)
    return out


def _exact_state(k, v, case, sink, comp):
    """The norms (and residual norms) that _state returns; its packed bytes are whole numbers."""
    out, m = [], case.get("qjl", 0)
    for x, bits in ((k, case["kbits"]), (v, case["vbits"])):
        if comp:
            n, _, _, _, gamma = _exact_codec(x[:, :, sink:sink + comp], bits, m)
            out += ([None, None] if bits != int(bits) else [None]) + [n] + ([None, gamma] if m else [])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":
        k, v, q = _generate_inputs(case, seed)
        outs, comp, res, sink, t = [], 0, 0, 0, 0
        for i, n in enumerate([case["prompt"]] + [1] * case["steps"]):
            a = min(case["sink"] - sink, n)
            sink, res, t = sink + a, res + n - a, t + n
            if res > 2 * case["window"]:
                comp, res = comp + res - case["window"], case["window"]
            if i:
                outs.append(_exact_attend(q[i - 1], *_exact_tokens(k[:, :, :t], v[:, :, :t], case, sink, comp)))
        return {"out": outs, "state": _exact_state(k, v, case, sink, comp)}
    if kind in ("decode", "dense"):
        g, outs = _gen(seed), []
        s, c, _ = _compressed(case, case["tokens"]) if kind == "decode" else (0, 0, 0)
        for _ in range(case["layers"]):
            k, v, q = _layer_inputs(case, g)
            k, v = _exact_tokens(k, v, case, s, c) if kind == "decode" else (k.double(), v.double())
            outs.append(_exact_attend(q, k, v))
        return outs
    if kind == "ragged":
        seqs, k1, v1, q = _ragged_inputs(case, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b, (k, v) in enumerate(seqs):
            k = torch.cat([k, k1[b][:, None]], dim=1)[None]
            v = torch.cat([v, v1[b][:, None]], dim=1)[None]
            s = min(k.shape[2], case["sink"])
            c = max(k.shape[2] - s - case["window"], 0)
            out[b] = _exact_attend(q[b:b + 1, :, None], *_exact_tokens(k, v, case, s, c))[0, :, 0]
        return [out]
    if kind in ("store", "fetch"):
        k, v = _kv(case, _gen(seed), case["batch"], case["tokens"])
        s, c, r = _compressed(case, case["tokens"])
        if kind == "fetch":
            return _exact_tokens(k, v, case, s, c)
        return _exact_state(k, v, case, s, c) + ([k[:, :, s + c:].double(), v[:, :, s + c:].double()] if r else [])
    if kind == "prefill":
        k, v, q = _layer_inputs(case, _gen(seed))
        s, c, _ = _compressed(case, case["tokens"])
        return _exact_attend(q, *_exact_tokens(k, v, case, s, c))
    x = _vectors(case, seed)
    n, corr, _, _, gamma = _exact_codec(x, case["bits"] - 1 if case["prod"] else case["bits"],
                                        case["d"] if case["prod"] else 0)
    return [None, n, corr, None, gamma] if case["prod"] else [None, n, corr]
