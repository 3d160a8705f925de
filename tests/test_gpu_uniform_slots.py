"""Blocks-per-wave instantiations 1 and 2 of the uniform-batch and fractional
kernels (up to 8 / 16 blocks of 32 tokens per workgroup): the boundary sizes,
against float64 over the stored codes at the kernels' bound."""

import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import min_cos, rel_err, to_dev
from test_gpu_attention import build, decode_route, dense_from_gpu_codes
from test_gpu_split import _geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kb,vb,route,G,blocks,tail,npw", [
    (4, 2, 2, 1, 32, 0, 1), (4, 2, 2, 4, 33, 31, 2), (4, 2, 2, 2, 65, 5, 4), (3, 4, 4, 8, 32, 3, 1), (3, 4, 4, 1, 64, 1, 2),
    (3.5, 2, 5, 2, 32, 0, 1), (3.5, 2, 5, 4, 33, 31, 2)])
def test_slots(kb, vb, route, G, blocks, tail, npw):
    """64 kv heads, 4 workgroups each: 8 / 9 / 16 / 17 blocks per workgroup."""
    H, window = 64, 16
    T = 32 * blocks - tail + window
    rng = np.random.RandomState(blocks + G)
    k, v = (rng.randn(1, H, T, 128).astype(np.float16) for _ in range(2))
    c, o = build(dict(head_dim=128, num_kv_heads=H, key_bits=kb, value_bits=vb, residual_window=window), k, v)
    q = rng.randn(1, H * G, 1, 128).astype(np.float16)
    qd = to_dev(q)
    assert decode_route(c, qd) == route
    assert _geometry(c, qd)[3] == npw
    out = c.attend(qd).cpu().numpy()
    kk, vv = dense_from_gpu_codes(c, o)
    ref = O.attention(q, kk, vv)
    assert rel_err(out, ref) < 5e-6 and min_cos(out, ref) >= 0.9999
    bf = c.attend(torch.from_numpy(q).to(torch.bfloat16).cuda()).cpu().numpy()  # the converted-query path
    ref = O.attention(torch.from_numpy(q).to(torch.bfloat16).double().numpy(), kk, vv)
    assert rel_err(bf, ref) < 5e-6
