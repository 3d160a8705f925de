"""bf16 and float32 queries past fp16's range (or with squares past float32's):
the decode kernels' query operands are fp16, scaled by a power of two per head.
One channel of every query is `big` and the scores' scale 2 / big, or the keys
that much smaller, so the logits are those of ordinary queries: float64
attention over the stored codes at 5e-6, the decode kernels' bound."""

import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import min_cos, rel_err, to_dev
from test_gpu_attention import build, decode_route, dense_from_gpu_codes
from test_gpu_mfma_decode import _caches, _kv

pytestmark = pytest.mark.gpu

BIG = [7e4, 1e5, 1.7e5, 1e6]  # 1.7e5: past fp16 where scale ||q|| of the default scale is not past the limit


def _query(shape, big, dtype, seed):
    q = np.random.RandomState(seed).randn(*shape)
    q[..., 5] = big
    q[:, 0, ..., 7] = -big  # head 0: two channels
    return torch.from_numpy(q).to(dtype).cuda()


def _held(got, q, k, v, scale):
    ref = O.attention(q.double().cpu().numpy(), k, v, scale)
    got = got.cpu().numpy()
    assert np.isfinite(got).all()
    assert rel_err(got, ref) < 5e-6 and min_cos(got, ref) >= 0.9999


@pytest.mark.parametrize("big", BIG + [1e22, 1e-22])
@pytest.mark.parametrize("D,kb,vb,m,G,dt,qdt", [
    (64, 4, 2, 0, 4, torch.bfloat16, torch.bfloat16), (96, 3, 3, 0, 5, torch.float16, torch.float32),
    (128, 4, 4, 0, 7, torch.bfloat16, torch.bfloat16), (256, 4, 3, 0, 4, torch.float16, torch.float32),
    (64, 3.5, 2.5, 32, 4, torch.bfloat16, torch.float32), (256, 4, 2, 32, 8, torch.float16, torch.bfloat16)])
def test_mfma_decode(D, kb, vb, m, G, dt, qdt, big):
    k, v = _kv(1, 2, 900, D, seed=D)
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, key_bits=kb, value_bits=vb, residual_window=64, fp16_sink_size=16,
                        **(dict(qjl_correction=True, qjl_n_proj=m) if m else {})), k, v, dt)
    q = _query((1, 2 * G, 1, D), big, qdt, D + G)
    assert decode_route(c, q) == 7
    kk, vv = dense_from_gpu_codes(c, o)
    _held(c.attend(q, scale=2 / big), q, kk, vv, 2 / big)


@pytest.mark.parametrize("big", BIG)
@pytest.mark.parametrize("D", [64, 256])
def test_mfma_decode_default_scale(D, big):
    """The default scale, the keys small instead."""
    k, v = _kv(1, 2, 900, D, seed=D, kmul=2 * D ** 0.5 / big)
    c, o = _caches(dict(head_dim=D, num_kv_heads=2, residual_window=64, fp16_sink_size=16), k, v, torch.bfloat16)
    q = _query((1, 8, 1, D), big, torch.float32, D)
    assert decode_route(c, q) == 7
    kk, vv = dense_from_gpu_codes(c, o)
    _held(c.attend(q), q, kk, vv, D ** -0.5)


@pytest.mark.parametrize("big", BIG)
@pytest.mark.parametrize("kb,vb,m,route", [(4, 2, 0, 2), (4, 2, 64, 3), (3, 4, 0, 4), (3.5, 2, 0, 5)])
@pytest.mark.parametrize("qdt", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_uniform_kernels(kb, vb, m, route, qdt, big):
    """Small keys (these kernels' rotated operands carry the scores' scale: one
    of 2e-6 would leave their fp16 remainders few bits)."""
    k, v = _kv(1, 2, 900, 128, seed=1, kmul=2 * 128 ** 0.5 / big)
    k, v = k.astype(np.float16), v.astype(np.float16)
    c, o = build(dict(head_dim=128, num_kv_heads=2, key_bits=kb, value_bits=vb, residual_window=64, fp16_sink_size=16,
                      **(dict(qjl_correction=True, qjl_n_proj=m) if m else {})), k, v)
    q = _query((1, 8, 1, 128), big, qdt, 2)
    assert decode_route(c, q) == route
    kk, vv = dense_from_gpu_codes(c, o)
    _held(c.attend(q), q, kk, vv, 128 ** -0.5)


@pytest.mark.parametrize("big", BIG)
@pytest.mark.parametrize("m", [0, 128])
def test_ragged_kernels(m, big):
    """Against the general kernel (float32 throughout)."""
    from turboquant_amd.ragged import RaggedKVBatch
    rb = RaggedKVBatch(2, 2, head_dim=128, key_bits=4, value_bits=2, residual_window=64, fp16_sink_size=16, qjl_n_proj=m)
    for b, t in enumerate((300, 1500)):
        rb.load(b, *(to_dev(x[0].astype(np.float16)) for x in _kv(1, 2, t, 128, seed=b, kmul=2 * 128 ** 0.5 / big)))
    q = _query((2, 8, 128), big, torch.bfloat16, 3)
    got = rb.attend(q).cpu().numpy()
    assert np.isfinite(got).all() and rel_err(got, rb.attend(q, general=True).cpu().numpy()) < 1e-5
