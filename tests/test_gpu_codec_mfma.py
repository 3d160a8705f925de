"""The MFMA codec kernels outside fp16 / head_dim 128 / no sketch: dequantize
(tq_dequant_mfma.hip) at the edges of its 32-token tiles, every width kind,
sketches and per-sequence spans, against float64 over the same codes; compress
(tq_compress_mfma.hip) against the oracle (codes outside the float32 boundary
band, bit-exact norms) and the general kernel."""

import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import code_parity, gpu_compress, rel_err, to_dev, unpack_codes

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _random_store(codec, B, H, T, seed):
    """A store of random codes (every code of both widths), norms and sketch."""
    from turboquant_amd import _codec
    st = _codec.PackedStore(codec, B, H, qjl=codec.qjl_m > 0)
    st.reserve(T, 0)
    g = torch.Generator(device=DEV).manual_seed(seed)
    for name in ("codes_hi", "codes_lo", "signs"):
        t = getattr(st, name)
        if t is not None:
            t.copy_(torch.randint(0, 256, t.shape, dtype=torch.uint8, device=DEV, generator=g))
    for name in ("norms", "gamma"):
        t = getattr(st, name)
        if t is not None:
            t.copy_(torch.exp(2 * torch.randn(t.shape, device=DEV, generator=g)))
    return st


def _exact(codec, st, bits, d, m):
    n = lambda t: None if t is None else t.cpu().numpy()
    x = O.dequantize(n(st.codes_hi), n(st.codes_lo), n(st.norms), O.rotation_matrix(d), bits, d)
    if m:
        signs = np.unpackbits(n(st.signs), axis=-1, bitorder="little").astype(bool)[..., :m]
        x = x + O.qjl_correction(signs, n(st.gamma), codec.proj.cpu().numpy()[:m], d)
    return x


@pytest.mark.parametrize("d,bits,m", [(64, 1, 0), (64, 3.5, 32), (96, 3, 96), (96, 2.5, 0), (128, 4, 0), (128, 2.5, 128),
                                      (128, 2, 40), (256, 4, 0), (256, 3.5, 32), (256, 2, 128)])
@pytest.mark.parametrize("n_b,src,dst", [([1, 1], [0, 0], [0, 0]), ([31, 33], [0, 5], [2, 0]), ([0, 300], [0, 1], [0, 7])])
def test_dequant_mfma(d, bits, m, n_b, src, dst):
    """Tokens src .. of each sequence to dst .. of the output, nothing else
    written; float64 over the codes at 5e-7 (operands to 2^-22, float32 sums)."""
    from turboquant_amd import _codec, _lib
    B, H, T = 2, 3, 320
    codec = _codec.get_codec(d, bits, 42, m, DEV)
    st = _random_store(codec, B, H, T, seed=d + m + n_b[1])
    out = torch.full((B, H, T, d), 7.0, device=DEV)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    nb, sb, db = i32(n_b), i32(src), i32(dst)
    span = _lib.Span(rows=B * H, heads=H, n_tok=max(n_b), reserved=0, n_tok_b=nb.data_ptr(), src_tok0_b=sb.data_ptr(),
                     dst_tok0_b=db.data_ptr())
    s = st.struct(0)
    _lib.check(_lib.load().tq_dequantize(codec.ref(), ctypes.byref(s), ctypes.byref(span), out.data_ptr(),
                                         out.stride(1), 1 if m else 0, _lib.stream_ptr(DEV)), "tq_dequantize")
    got, ref = out.cpu().numpy(), _exact(codec, st, bits, d, m)
    for b in range(B):
        x = got[b, :, dst[b]:dst[b] + n_b[b]]
        if n_b[b]:
            assert rel_err(x, ref[b, :, src[b]:src[b] + n_b[b]]) < 5e-7
        rest = np.delete(got[b], np.s_[dst[b]:dst[b] + n_b[b]], axis=1)
        assert (rest == 7.0).all()


def _compress(x, bits, m=0, general=False):
    """numpy (codes_hi, codes_lo, norms, signs, gamma) of a (B, H, T, D) tensor."""
    from turboquant_amd import _codec
    B, H, T, D = x.shape
    codec = _codec.get_codec(D, bits, 42, m, x.device)
    st = _codec.PackedStore(codec, B, H, qjl=m > 0)
    st.reserve(T, 0)
    _codec.compress_into(codec, x, 0, T, st, 0, general=general)
    return tuple(None if t is None else t[:, :, :T].cpu().numpy()
                 for t in (st.codes_hi, st.codes_lo, st.norms, st.signs, st.gamma))


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("d,bits", [(64, 1), (64, 3.5), (64, 4), (96, 3), (96, 2), (128, 4), (128, 2.5), (128, 1),
                                    (256, 4), (256, 3.5), (256, 2)])
@pytest.mark.parametrize("T", [1, 63, 65, 700])
def test_compress_mfma_codes(d, bits, dt, T):
    rng = np.random.RandomState(int(d + 10 * bits + T))
    x = torch.from_numpy(rng.randn(2, 3, T, d).astype(np.float32) * np.exp(rng.randn(2, 3, T, 1)).astype(np.float32)).to(dt)
    xf = x.float().numpy()
    _, _, _, _, norms_equal, _ = code_parity(xf, bits, gpu=_compress(x.cuda(), bits))
    assert norms_equal


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("d,bits,m", [(64, 2, 64), (96, 3, 32), (128, 4, 128), (128, 3.5, 40), (128, 1, 96)])
def test_compress_mfma_sketch(d, bits, m, dt):
    """Signs of projections away from zero (|r . S| > 1e-4 ||x||; the residual
    and its projection carry about 1e-6 ||x||) and residual norms, float64 over
    the kernel's own codes."""
    rng = np.random.RandomState(d + m)
    x = torch.from_numpy(rng.randn(1, 2, 150, d).astype(np.float32)).to(dt)
    hi, lo, n, signs, gamma = _compress(x.cuda(), bits, m)
    xf = x.double().numpy()
    code_parity(x.float().numpy(), bits, gpu=(hi, lo, n, None, None))
    res = xf - O.dequantize(hi, lo, n, O.rotation_matrix(d), bits, d)
    from turboquant_amd.qjl import generate_projection_matrix
    proj = res @ generate_projection_matrix(d, m).astype(np.float64).T
    got = np.unpackbits(signs, axis=-1, bitorder="little").astype(bool)
    clear = np.abs(proj) > 1e-4 * np.linalg.norm(xf, axis=-1, keepdims=True)
    assert clear.mean() > 0.9 and (got[..., :m] == (proj >= 0))[clear].all()
    assert got[..., m:].all()  # the zero rows past m project to 0: bit set
    assert rel_err(gamma, np.linalg.norm(res, axis=-1)) < 2e-6


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("d", [64, 96, 128, 256])
def test_compress_mfma_special_vectors(d, dt):
    """Zero, tiny, subnormal, huge, overflowing-norm, infinite and NaN vectors:
    the codes and norms of the general kernel."""
    rng = np.random.RandomState(d)
    base = torch.from_numpy(rng.randn(16, d).astype(np.float32))
    mul = {torch.float16: [1, 0, 6e-8, 1e-6, 1e4], torch.bfloat16: [1, 0, 1e-40, 1e-36, 1e-20, 1e30, 3e37],
           torch.float32: [1, 0, 1e-42, 1e-37, 1e-20, 1e30, 3e37, 1e38]}[dt]
    rows = [base * f for f in mul]
    rows += [base.index_fill(1, torch.tensor([3]), v) for v in (float("inf"), float("-inf"), float("nan"))]
    x = torch.cat(rows).clamp(-3.3e38, 3.3e38) if dt == torch.float32 else torch.cat(rows)
    x = torch.cat([x, *(base.index_fill(1, torch.tensor([3]), float("inf")),)]).to(dt)[None, None].cuda().contiguous()
    for bits in (4, 1):
        a, b = _compress(x, bits), _compress(x, bits, general=True)
        assert np.array_equal(a[2], b[2], equal_nan=True)
        ca, cb = unpack_codes(a[0], a[1], bits, d), unpack_codes(b[0], b[1], bits, d)
        bad = (ca != cb).any(-1)[0, 0]
        assert not bad.any(), (np.nonzero(bad)[0] // 16, bits)


@pytest.mark.parametrize("d,bits,m", [(64, 3.5, 32), (96, 3, 0), (128, 4, 128), (256, 2, 0)])
def test_dequant_mfma_small_norms(d, bits, m):
    """Norms from 1 down to 1e-36 (and as far up): each vector to float32 rounding. 5e-7 of its own norm, as above:
    the coordinates are normal float32 numbers down to 1e-38, a few of them below that are exact to 1e-45."""
    from turboquant_amd import _codec
    codec = _codec.get_codec(d, bits, 42, m, DEV)
    st = _random_store(codec, 1, 2, 80, seed=d)
    st.norms[:, 0, :80] = 10.0 ** torch.linspace(0, -36, 80, device=DEV)
    st.norms[:, 1, :80] = 10.0 ** torch.linspace(0, 36, 80, device=DEV)
    if m:
        st.gamma.copy_(st.norms * 0.3)
    out = torch.empty(1, 2, 80, d, device=DEV)
    _codec.dequantize_into(codec, st, 0, 80, out, 0, m > 0)
    got, ref = out.double().cpu().numpy(), _exact(codec, st, bits, d, m)[:, :, :80]
    assert (np.linalg.norm(got - ref, axis=-1) < 5e-7 * np.linalg.norm(ref, axis=-1)).all()


@pytest.mark.parametrize("d", [64, 96, 128, 256])
def test_compress_mfma_norm_at_the_end_of_float32(d):
    """Vectors along a row of R whose norm is float32's largest value or a few units below: the rotated coordinate may
    pass it (the quantizer's cells are looked up inside the table). Codes of the general kernel, which divides first."""
    R = O.rotation_matrix(d).astype(np.float64)
    top = float(np.finfo(np.float32).max)
    f = np.array([1 - k * 2.0 ** -24 for k in (0, 1, 2, 3, 4, 8, 1 << 20)])
    x = (np.concatenate([R, -R])[:, None] * (f[:, None] * top)).astype(np.float32).reshape(1, 1, -1, d)
    x = torch.from_numpy(x).cuda()
    for bits in (4, 2):
        a, b = _compress(x, bits), _compress(x, bits, general=True)
        assert np.array_equal(a[2], b[2]) and np.isfinite(b[2]).mean() > 0.5
        ca, cb = unpack_codes(a[0], a[1], bits, d), unpack_codes(b[0], b[1], bits, d)
        big = np.abs(x.cpu().double().numpy() @ R.T) > 1e38  # (the others are 0 up to rounding: a cell boundary)
        fin = np.isfinite(b[2])[..., None] & big
        assert (ca == cb)[fin].all()
