"""GPU parity of the decode kernels of tq_decode_mfma.h: head_dim 64 / 96 /
128 / 256, integer and fractional widths on either side, any number of query
heads per kv head, fp16 and bf16 uncompressed tokens, uniform and ragged
batches. The route is asserted through the library's test hook (7), the
output held to float64 attention over the stored codes at 5e-6 (scores and
weights carry about 2^-22 relative, as in the K4/V2 kernels' bound) and to the
general kernel at 1e-4.
"""

import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import min_cos, rel_err, to_dev
from test_gpu_attention import decode_route, dense_from_gpu_codes

pytestmark = pytest.mark.gpu

REL_TOL = 5e-6
COS_TOL = 0.9999


def _kv(B, H, T, D, seed, kmul=1.0, vmul=1.0):
    rng = np.random.RandomState(seed)
    s = np.exp(rng.randn(D) * 0.5)
    return (rng.randn(B, H, T, D) * s * kmul).astype(np.float32), (rng.randn(B, H, T, D) * vmul).astype(np.float32)


def _caches(kw, k, v, dt):
    from turboquant_amd import TurboQuantKVCache
    kt, vt = torch.from_numpy(k).to(dt), torch.from_numpy(v).to(dt)
    c = TurboQuantKVCache(**kw)
    c.update(kt.cuda(), vt.cuda())
    o = O.CacheOracle(**kw)
    o.update(kt.float().numpy(), vt.float().numpy())
    return c, o


def _check(c, o, q, label, route=7):
    qd = to_dev(q)
    assert decode_route(c, qd) == route
    fast = c.attend(qd).cpu().numpy()
    gen = c.attend(qd, general_kernel=True).cpu().numpy()
    kk, vv = dense_from_gpu_codes(c, o)
    ref = O.attention(q, kk, vv)
    print(f"{label}: rel {rel_err(fast, ref):.3e} vs general {rel_err(fast, gen):.3e}")
    assert np.isfinite(fast).all()
    assert rel_err(fast, ref) < REL_TOL and min_cos(fast, ref) >= COS_TOL
    assert rel_err(fast, gen) < 1e-4


PAIRS = [(4, 2), (2, 4), (3, 3), (4, 4), (3.5, 2.5), (2.5, 3.5), (3, 2.5)]


@pytest.mark.parametrize("D,kb,vb", [(d, k, v) for d in (64, 96, 256) for k, v in PAIRS if d != 96 or k == int(k)] + [
    (128, 4, 4), (128, 3.5, 2)], ids=str)
@pytest.mark.parametrize("G,T,sink,window,dt", [
    (4, 1500, 16, 64, torch.bfloat16),  # a partial last block, one workgroup's uncompressed tokens
    (7, 700, 0, 32, torch.float16),     # eight columns with an idle one
    (1, 9000, 300, 300, torch.bfloat16),  # several blocks per wave, three workgroups of uncompressed tokens
])
def test_mfma_matches_oracle(D, kb, vb, G, T, sink, window, dt):
    if D == 128 and dt == torch.float16 and G != 7:
        pytest.skip("another route")
    k, v = _kv(1, 2, T, D, seed=int(T + 10 * kb + vb + G))
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, key_bits=kb, value_bits=vb, residual_window=window,
                        fp16_sink_size=sink), k, v, dt)
    q = np.random.RandomState(int(kb * 8 + vb + G)).randn(1, 2 * G, 1, D).astype(np.float16)
    _check(c, o, q, f"d{D} K{kb}/V{vb} G={G} T={T} {dt}")


@pytest.mark.parametrize("D,G,batch", [(128, 3, 2), (64, 16, 1), (256, 10, 1), (96, 12, 3), (128, 5, 1)])
def test_mfma_query_groups(D, G, batch):
    """Head groups of at most 8 per launch row: 3, 8 + 8, 5 + 5, 6 + 6, 5."""
    k, v = _kv(batch, 2, 1000, D, seed=D + G)
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, residual_window=64, fp16_sink_size=4), k, v, torch.float16)
    q = np.random.RandomState(G).randn(batch, 2 * G, 1, D).astype(np.float16)
    _check(c, o, q, f"d{D} G={G} B={batch}")


@pytest.mark.parametrize("D,T", [(64, 1), (64, 33), (96, 200), (256, 256)])
def test_mfma_uncompressed_only(D, T):
    k, v = _kv(2, 2, T, D, seed=T)
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, residual_window=128, fp16_sink_size=16), k, v, torch.bfloat16)
    assert c._compressed_len == 0
    _check(c, o, np.random.RandomState(T).randn(2, 8, 1, D).astype(np.float16), f"d{D} T={T}")


# (a score of magnitude S is exact to about S 2^-22, so its weight to that
# relative error: 5e-6 holds for |S| up to about 20, logits of std 1.5 here)
@pytest.mark.parametrize("kmul,vmul,qmul", [(300.0, 3e4, 1.0), (1e-3, 1e-7, 1.0), (1.0, 1.0, 1e-5)])
@pytest.mark.parametrize("D", [64, 256])
def test_mfma_magnitudes(D, kmul, vmul, qmul):
    """bf16 tokens past / below the fp16 range, queries whose fp16 operands
    need a power of two, value norms that move the weights' exponent."""
    k, v = _kv(1, 2, 900, D, seed=3, kmul=kmul, vmul=vmul)
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, residual_window=64, fp16_sink_size=16), k, v, torch.bfloat16)
    q = (np.random.RandomState(1).randn(1, 8, 1, D) * qmul / kmul).astype(np.float32)
    _check(c, o, q, f"d{D} k x{kmul} v x{vmul} q x{qmul}")


def _one_sequence(d, b, H, q, out):
    """Descriptor d with sequence b of its batch alone (same stores, sink and ring)."""
    one = type(d).from_buffer_copy(d)
    one.batch, one.q, one.out = 1, q.data_ptr(), out.data_ptr()
    for st in (one.kstore, one.vstore):
        for name, stride, size in (("codes_hi", st.hi_head_stride, 1), ("codes_lo", st.lo_head_stride, 1), ("norms", st.norm_head_stride, 4),
                                   ("signs", st.sign_head_stride, 1), ("gamma", st.gamma_head_stride, 4)):
            if getattr(st, name):
                setattr(st, name, getattr(st, name) + b * H * stride * size)
    for name, stride in (("sink_k", d.sink_head_stride), ("sink_v", d.sink_head_stride), ("res_k", d.res_head_stride),
                         ("res_v", d.res_head_stride)):
        setattr(one, name, getattr(one, name) + b * H * stride * 2)
    for name in ("comp_len", "sink_len", "res_len", "res_start"):
        setattr(one, name, getattr(one, name) + 4 * b)
    return one


@pytest.mark.parametrize("D,kb,vb,m,G,bf", [(128, 3.5, 3, 0, 3, False), (128, 3, 3, 32, 4, False), (64, 4, 2, 0, 4, True),
                                            (256, 4, 3, 0, 2, True), (256, 4, 2, 32, 8, False), (64, 3.5, 2.5, 32, 7, True)])
def test_mfma_ragged_equals_single_sequences(D, kb, vb, m, G, bf):
    """A ragged batch (per-sequence lengths, a sequence with nothing
    compressed, wrapped rings) on these kernels: each sequence equals its own
    call over the same stores, whose partials are cut elsewhere, and float64
    attention over what is stored."""
    from turboquant_amd import _lib
    from turboquant_amd.ragged import RaggedKVBatch
    H = 2
    lens = [40, 300, 1777, 5000]
    rb = RaggedKVBatch(4, H, head_dim=D, key_bits=kb, value_bits=vb, residual_window=64, fp16_sink_size=16, qjl_n_proj=m)
    rng = np.random.RandomState(9)
    for b, t in enumerate(lens):
        rb.load(b, *(to_dev(rng.randn(H, t, D).astype(np.float16)) for _ in range(2)))
    for _ in range(5):
        rb.step(*(to_dev(rng.randn(4, H, D).astype(np.float16)) for _ in range(2)))
    assert rb.comp_len[0] == 0 and (rb.res_start[1:] + rb.res_len[1:] > rb.cap).all()
    q = to_dev(rng.randn(4, H * G, D).astype(np.float16))
    out = torch.empty(q.shape, dtype=torch.float32, device=q.device)
    d, keep = rb.descriptor(q, out, D ** -0.5)
    d = type(d).from_buffer_copy(d)  # (the batch refreshes its own for every call)
    sink_k, sink_v, ring_k, ring_v = rb.sink_k, rb.sink_v, rb.ring_k, rb.ring_v
    if bf:
        sink_k, sink_v, ring_k, ring_v = (t.bfloat16() for t in (sink_k, sink_v, ring_k, ring_v))
        d.kv_dtype = _lib.TQ_BF16
        d.sink_k, d.sink_v, d.res_k, d.res_v = (t.data_ptr() for t in (sink_k, sink_v, ring_k, ring_v))
    lib = _lib.load()
    fn = lib.tq_debug_decode_route
    fn.restype, fn.argtypes = ctypes.c_int32, [ctypes.c_void_p] * 3

    def call(desc):
        assert fn(ctypes.addressof(rb.kc.struct), ctypes.addressof(rb.vc.struct), ctypes.addressof(desc)) == 7
        need = lib.tq_attention_workspace_bytes(rb.kc.ref(), rb.vc.ref(), ctypes.byref(desc))
        ws = torch.empty(need, dtype=torch.uint8, device=q.device)
        _lib.check(lib.tq_decode_attention(rb.kc.ref(), rb.vc.ref(), ctypes.byref(desc), ws.data_ptr(), need,
                                           _lib.stream_ptr(q.device)), "tq_decode_attention")
        torch.cuda.synchronize()

    call(d)
    got = out.cpu().numpy()
    if not bf:
        assert np.array_equal(got, rb.attend(q).cpu().numpy())
        gen = rb.attend(q, general=True).cpu().numpy()
    R = O.rotation_matrix(D)
    n64 = lambda t: t.cpu().double().numpy()
    for b in range(4):
        qb, ob = q[b:b + 1].contiguous(), torch.empty(1, H * G, D, device=q.device)
        call(_one_sequence(d, b, H, qb, ob))
        assert rel_err(got[b:b + 1], ob.cpu().numpy()) < 2e-6, b
        C, S = int(rb.comp_len[b]), int(rb.sink_len[b])
        slots = torch.as_tensor((rb.res_start[b] + np.arange(rb.res_len[b])) % rb.cap, device=q.device)
        dense = []
        for st, codec, sk, ring in ((rb.kstore, rb.kc, sink_k, ring_k), (rb.vstore, rb.vc, sink_v, ring_v)):
            seg = [n64(sk[b:b + 1, :, :S])]
            if C:
                part = lambda t: None if t is None else t[b:b + 1, :, :C].cpu().numpy()
                x = O.dequantize(part(st.codes_hi), part(st.codes_lo), part(st.norms), R, codec.bits, D)
                if m:
                    signs = np.unpackbits(part(st.signs), axis=-1, bitorder="little").astype(bool)
                    x = x + O.qjl_correction(signs, part(st.gamma), rb.kc.proj.cpu().numpy(), D)
                seg.append(x)
            dense.append(np.concatenate(seg + [n64(ring[b:b + 1][:, :, slots])], axis=2))
        ref = O.attention(n64(qb)[:, :, None], *dense)[:, :, 0]
        assert rel_err(got[b:b + 1], ref) < REL_TOL and min_cos(got[b:b + 1], ref) >= COS_TOL, b
        if not bf:
            assert rel_err(got[b], gen[b]) < REL_TOL, b


def test_mfma_more_than_256_partials():
    """A residual window of 70,000 tokens: 274 workgroups of uncompressed tokens beside those of the compressed ones,
    more headers than the merge holds in registers."""
    T, W = 73000, 70000
    k, v = _kv(1, 1, T, 64, seed=1)
    c, o = _caches(dict(head_dim=64, num_kv_heads=1, residual_window=W, chunk_size=1, fp16_sink_size=8), k, v, torch.bfloat16)
    assert c._compressed_len == T - W - 8
    _check(c, o, np.random.RandomState(4).randn(1, 4, 1, 64).astype(np.float16), "window 70000")


def test_mfma_ten_million_tokens():
    """An uncompressed list whose partials, one per 256 tokens, would pass the merge's LDS (a launch that fails is an error
    too, not a call without output): the general kernel's result."""
    from turboquant_amd import TurboQuantKVCache
    T = 9_600_000
    g = torch.Generator(device="cuda").manual_seed(1)
    k, v = (torch.randn(1, 1, T, 64, generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    c = TurboQuantKVCache(head_dim=64, num_kv_heads=1, residual_window=T, chunk_size=1)
    c.update(k, v)
    q = torch.randn(1, 2, 1, 64, generator=g, device="cuda")
    assert c._compressed_len == 0 and decode_route(c, q) == 7
    got, gen = c.attend(q), c.attend(q, general_kernel=True)
    # 9.6M weights of one part each: the sums carry float32 rounding of their order, 1e-5 of the small average
    assert (got - gen).norm() < 1e-4 * gen.norm()


@pytest.mark.parametrize("D,kb,vb,m,dt", [(64, 4, 2, 0, torch.bfloat16), (256, 4, 3, 32, torch.float16)])
def test_mfma_no_allocation_entry(D, kb, vb, m, dt):
    """tq_decode_attention_noalloc on these kernels: bit-equal to the workspace entry point, eager (a smaller call over
    the scratch of a larger one) and captured, replayed with eager calls on the same scratch between."""
    from turboquant_amd import _lib
    lib = _lib.load()
    calls = []
    for T, seed in ((3000, 1), (700, 2)):
        k, v = _kv(1, 2, T, D, seed=seed)
        c, _ = _caches(dict(head_dim=D, num_kv_heads=2, key_bits=kb, value_bits=vb, residual_window=64, fp16_sink_size=16,
                            **(dict(qjl_correction=True, qjl_n_proj=m) if m else {})), k, v, dt)
        q = to_dev(np.random.RandomState(seed).randn(1, 8, 1, D).astype(np.float16))
        assert decode_route(c, q) == 7
        calls.append((c, q, c.attend(q)))

    def noalloc(c, q, out):
        desc = c.attention_descriptor(q, out, D ** -0.5)
        _lib.check(lib.tq_decode_attention_noalloc(c._kc.ref(), c._vc.ref(), ctypes.byref(desc), _lib.stream_ptr(q.device)),
                   "tq_decode_attention_noalloc")

    for c, q, ref in calls:
        out = torch.full_like(ref, float("nan"))
        noalloc(c, q, out)
        assert torch.equal(out, ref)
    (c, q, ref), (c2, q2, ref2) = calls
    out = torch.empty_like(ref)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        noalloc(c, q, out)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        out2 = torch.full_like(ref2, float("nan"))
        noalloc(c2, q2, out2)
        torch.cuda.synchronize()
        assert torch.equal(out2, ref2)


def test_mfma_graph_replays():
    """Captured and replayed several times with eager work between: the same
    output as the eager call."""
    k, v = _kv(1, 2, 2000, 64, seed=8)
    c, _ = _caches(dict(head_dim=64, num_kv_heads=2, residual_window=64), k, v, torch.bfloat16)
    q = to_dev(np.random.RandomState(2).randn(1, 8, 1, 64).astype(np.float16))
    ref = c.attend(q).clone()
    out = torch.empty_like(ref)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        c.attend(q, out=out)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        c.attend(q, out=out)
    for _ in range(4):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        assert torch.equal(c.attend(q), ref)


@pytest.mark.parametrize("D,kb,vb,m,G,T,dt", [
    (64, 4, 2, 32, 4, 1500, torch.bfloat16), (64, 3.5, 2.5, 7, 7, 300, torch.float16), (96, 3, 3, 32, 1, 5000, torch.float16),
    (128, 3, 3, 32, 4, 700, torch.bfloat16), (128, 4, 3.5, 20, 8, 9000, torch.float16), (128, 4, 2, 32, 5, 1000, torch.float16),
    (256, 4, 3, 32, 2, 1500, torch.bfloat16), (256, 2, 2, 32, 10, 400, torch.float16)])
def test_mfma_sketch(D, kb, vb, m, G, T, dt):
    """The two terms of a sketch of at most 32 projections."""
    k, v = _kv(1, 2, T, D, seed=T + D)
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, key_bits=kb, value_bits=vb, residual_window=64, fp16_sink_size=16,
                        qjl_correction=True, qjl_n_proj=m), k, v, dt)
    q = np.random.RandomState(G).randn(1, 2 * G, 1, D).astype(np.float16)
    _check(c, o, q, f"QJL d{D} K{kb}/V{vb} m={m} G={G} T={T}")


def test_mfma_sketch_gammas_past_the_norms():
    """Residual norms far above (and below) the value norms, as a loaded state
    may hold: the weights' exponent follows the larger of the two."""
    k, v = _kv(1, 2, 900, 64, seed=5)
    c, o = _caches(dict(head_dim=64, num_kv_heads=2, residual_window=64, qjl_correction=True, qjl_n_proj=32), k, v,
                   torch.float16)
    q = np.random.RandomState(3).randn(1, 8, 1, 64).astype(np.float16)
    for f in (3e4, 1e-4):
        c._vstore.gamma.mul_(f)
        _check(c, o, q, f"gamma x{f}")


@pytest.mark.parametrize("D,kb,vb,G,dt,m", [(64, 4, 2, 4, torch.bfloat16, 0), (128, 3.5, 3, 7, torch.float16, 0),
                                            (256, 4, 3, 4, torch.bfloat16, 0), (96, 3, 3, 2, torch.float16, 32)])
@pytest.mark.parametrize("what", ["query NaN", "query inf", "norm NaN", "norm inf", "ring key NaN", "value norm NaN"])
def test_mfma_non_finite(D, kb, vb, G, dt, m, what):
    """A NaN in a query, a stored norm or a ring key takes the whole head, not one workgroup's tokens: the general
    kernel's output (zeros where the weights' sum is NaN), the other heads as without it."""
    k, v = _kv(1, 2, 3000, D, seed=D)
    c, _ = _caches(dict(head_dim=D, num_kv_heads=2, key_bits=kb, value_bits=vb, residual_window=64, fp16_sink_size=16,
                        **(dict(qjl_correction=True, qjl_n_proj=m) if m else {})), k, v, dt)
    q = to_dev(np.random.RandomState(G).randn(1, 2 * G, 1, D).astype(np.float16))
    clean = c.attend(q).cpu().numpy()
    bad = float("inf") if "inf" in what else float("nan")
    hit = slice(0, G)
    if "query" in what:
        q[0, 1, 0, 3] = bad
        hit = slice(1, 2)
    elif what.startswith("norm"):
        c._kstore.norms[0, 0, 1500] = bad
    elif what.startswith("value"):
        c._vstore.norms[0, 0, 1500] = bad
    else:
        c._res_k[0, 0, (c._res_start + 5) % c._res_cap, 3] = bad
    assert decode_route(c, q) == 7
    got, gen = c.attend(q).cpu().numpy(), c.attend(q, general_kernel=True).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(gen)) and np.isnan(gen).any() == (what == "value norm NaN")
    if "NaN" in what:
        assert not np.nan_to_num(got[:, hit]).any()
    assert rel_err(np.nan_to_num(got), np.nan_to_num(gen)) < 1e-4
    rest = np.delete(got, hit, axis=1)
    assert np.isfinite(rest).all() and np.array_equal(rest, np.delete(clean, hit, axis=1))


@pytest.mark.parametrize("D,G,dt,T", [(64, 4, torch.bfloat16, 2000), (128, 7, torch.float16, 300), (256, 2, torch.float16, 900),
                                      (96, 8, torch.bfloat16, 700), (64, 12, torch.float16, 200)])
@pytest.mark.parametrize("what", ["value inf", "value -inf", "key", "both"])
def test_mfma_infinite_tokens(D, G, dt, T, what):
    """Infinite elements of uncompressed tokens, in the sink, at the start and at the end of the ring: a value's dim is
    that infinity and the others stay; a key whose score is -inf has no weight, one of +inf makes the head zero."""
    k, v = _kv(1, 2, T, D, seed=D)
    c, _ = _caches(dict(head_dim=D, num_kv_heads=2, residual_window=150, fp16_sink_size=16), k, v, dt)
    q = to_dev(np.abs(np.random.RandomState(G).randn(1, 2 * G, 1, D)).astype(np.float16))
    q[0, 2, 0] *= -1  # the other sign of an infinite score
    inf = float("inf")
    end = (c._res_start + c._fp16_len - 1) % c._res_cap
    if what != "key":
        x = -inf if "-" in what else inf
        c.sink_values[0, 0, 3, 7] = x
        c._res_v[0, 1, c._res_start, 0] = x
        c._res_v[0, 1, end, D - 1] = -x
    if what in ("key", "both"):
        c.sink_keys[0, 0, 15, 2] = -inf
        c._res_k[0, 1, end, D // 2] = -inf
    assert decode_route(c, q) == 7
    got, gen = c.attend(q).cpu().numpy(), c.attend(q, general_kernel=True).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(gen))
    assert np.array_equal(got[np.isinf(gen)], gen[np.isinf(gen)]) and np.isinf(gen).any() == (what != "key")
    f = np.isfinite(gen)
    assert np.isfinite(got[f]).all() and rel_err(got[f], gen[f]) < 1e-4
    assert f.mean() > 0.9 or what == "both"


@pytest.mark.parametrize("D,m", [(64, 0), (128, 32)])
@pytest.mark.parametrize("vmul", [1e-36, 1e33])
def test_mfma_value_norms(D, m, vmul):
    """Value norms near float32's ends, alone and in every other block of each wave beside ordinary ones (15 workgroups a
    row, 14 or more blocks each): the weights' exponent covers them (1e-36 times a weight is normal down to 1e-2 of the
    largest, below that exact to 1e-45: 2e-7 of an output; 1e33 leaves room for the general kernel's unscaled sums)."""
    T = 6800
    odd = np.arange(T)[:, None] // 256 % 2 == 1
    for H, n, mul in ((2, 900, vmul), (16, T, np.where(odd, vmul, 1.0)), (16, T, np.where(odd, 1.0, vmul))):
        k, v = _kv(1, H, n, D, seed=3)
        q = np.random.RandomState(1).randn(1, H, 1, D).astype(np.float32)
        c, o = _caches(dict(head_dim=D, num_kv_heads=H, residual_window=64, fp16_sink_size=16, key_bits=4, value_bits=3,
                            **(dict(qjl_correction=True, qjl_n_proj=m) if m else {})), k, v * mul, torch.bfloat16)
        _check(c, o, q, f"d{D} v x{vmul}")


@pytest.mark.parametrize("hkv,G,batch,tokens,route", [
    (8, 4, 1, 131072, 7), (8, 4, 8, 16384, 7), (8, 4, 8, 32768, 3), (8, 8, 8, 32768, 7), (8, 1, 3, 8192, 7), (8, 1, 2, 131072, 7), (8, 2, 4, 65536, 3),
    (8, 4, 16, 4096, 7), (8, 4, 16, 8192, 3), (8, 4, 12, 10923, 3), (8, 4, 32, 4096, 7), (4, 4, 64, 8192, 3),
    (8, 3, 16, 16384, 7), (16, 16, 16, 16384, 7)])
def test_sketch_route_by_size(hkv, G, batch, tokens, route):
    """K4/V2 with 32 projections: the K4/V2 kernels where the mfma grid would leave CUs idle for long, if they take the
    ratio (a descriptor of that size over a small cache; nothing is launched)."""
    from turboquant_amd import _lib
    k, v = _kv(1, hkv, 100, 128, seed=0)
    c, _ = _caches(dict(head_dim=128, num_kv_heads=hkv, residual_window=16, qjl_correction=True, qjl_n_proj=32), k, v,
                   torch.float16)
    q = torch.zeros(1, hkv * G, 128, device="cuda", dtype=torch.float16)
    d = c.attention_descriptor(q, torch.empty(q.shape, device="cuda"), 0.1)
    d.batch, d.max_comp, d.max_res = batch, tokens - 128, 128
    fn = _lib.load().tq_debug_decode_route
    fn.restype, fn.argtypes = ctypes.c_int32, [ctypes.c_void_p] * 3
    assert fn(ctypes.addressof(c._kc.struct), ctypes.addressof(c._vc.struct), ctypes.addressof(d)) == route


@pytest.mark.parametrize("G,T,route", [(4, 3520, 7), (1, 3521, 3)])
def test_sketch_both_routes(G, T, route):
    """Either side of that line (88 rows: 110 blocks)."""
    k, v = _kv(11, 8, T + 40, 128, seed=T)
    c, o = _caches(dict(head_dim=128, num_kv_heads=8, residual_window=40, chunk_size=1, qjl_correction=True, qjl_n_proj=32),
                   k, v, torch.float16)
    assert c._compressed_len == T
    _check(c, o, np.random.RandomState(G).randn(11, 8 * G, 1, 128).astype(np.float16), f"QJL G={G} T={T}", route)


@pytest.mark.parametrize("D,m", [(64, 0), (256, 32)])
def test_mfma_rotation_parts_of_two_planes(D, m):
    """A key codec without the third plane's flag: the remainder of [1], the same bound."""
    from turboquant_amd import _lib
    k, v = _kv(1, 2, 1500, D, seed=D)
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, residual_window=64, fp16_sink_size=16,
                        **(dict(qjl_correction=True, qjl_n_proj=m) if m else {})), k, v, torch.bfloat16)
    q = np.random.RandomState(3).randn(1, 8, 1, D).astype(np.float16)
    qd = to_dev(q)
    three = c.attend(qd).cpu().numpy()
    two = _lib.Codec.from_buffer_copy(c._kc.struct)
    assert two.flags & _lib.TQ_CODEC_ROTATION_LO2
    two.flags = 0
    out = torch.empty(1, 8, 1, D, device="cuda")
    d = c.attention_descriptor(qd, out, D ** -0.5)
    lib = _lib.load()
    need = lib.tq_attention_workspace_bytes(ctypes.byref(two), c._vc.ref(), ctypes.byref(d))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    _lib.check(lib.tq_decode_attention(ctypes.byref(two), c._vc.ref(), ctypes.byref(d), ws.data_ptr(), need,
                                       _lib.stream_ptr(out.device)), "tq_decode_attention")
    got = out.cpu().numpy()
    ref = O.attention(q, *dense_from_gpu_codes(c, o))
    assert not np.array_equal(got, three) and rel_err(got, ref) < REL_TOL and rel_err(three, ref) < REL_TOL
