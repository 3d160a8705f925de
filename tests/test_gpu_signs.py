"""Sketch sign rows to bools and back (tq_unpack_signs / tq_pack_signs): exact, at the edges of the 16- and
32-projection pieces, with rows past one grid and misaligned bool rows."""

import numpy as np
import pytest
import torch

from turboquant_amd import _lib
from turboquant_amd.quantizer import _pack_signs, _unpack_signs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 48, 100, 128, 255, 256])
@pytest.mark.parametrize("n", [1, 7, 4099])
@pytest.mark.parametrize("offset", [0, 1])
def test_signs_round_trip(m, n, offset):
    rng = np.random.default_rng(m * 1000 + n)
    mp = (m + 31) // 32 * 32
    signs = rng.integers(0, 2, (n, m)).astype(bool)
    padded = np.zeros((n, mp), bool)
    padded[:, :m] = signs
    want = np.packbits(padded, axis=-1, bitorder="little")
    buf = torch.empty(n * m + offset, dtype=torch.bool, device="cuda")
    dev = buf[offset:].view(n, m)
    dev.copy_(torch.from_numpy(signs))
    rows = _pack_signs(dev, mp)
    assert np.array_equal(rows.cpu().numpy(), want)
    assert np.array_equal(_pack_signs(dev.to(torch.int32), mp).cpu().numpy(), want)  # other types: torch operators
    # padding bits are not read
    noisy = want | np.packbits(~padded & (np.arange(mp) >= m), axis=-1, bitorder="little")
    got = _unpack_signs(torch.from_numpy(noisy).cuda(), m)
    assert got.dtype == torch.bool and np.array_equal(got.cpu().numpy(), signs)
    guard = torch.full((n * m + offset + 1,), 7, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.load().tq_unpack_signs(rows.data_ptr(), n, m, mp // 8, guard[offset:].data_ptr(),
                                           _lib.stream_ptr(guard.device)), "unpack_signs")
    g = guard.cpu().numpy()
    assert np.array_equal(g[offset:-1].reshape(n, m), signs) and g[-1] == 7 and (offset == 0 or g[0] == 7)


def test_rows_past_one_grid():
    n, m = 16384 * 256 // 8 + 77, 128
    signs = torch.randint(0, 2, (n, m), device="cuda", dtype=torch.uint8).bool()
    assert torch.equal(_unpack_signs(_pack_signs(signs, m), m), signs)
