"""The MFMA codec kernels outside fp16 / head_dim 128 / no sketch: dequantize
(tq_dequant_mfma.hip) at the edges of its 32-token tiles, every width kind,
sketches and per-sequence spans, against float64 over the same codes."""

import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import rel_err, to_dev

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
