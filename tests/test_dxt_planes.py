"""The DXT encoder keeps a block's channels as planes of four texels to a word.
Its byte range (16-bit minima of a word as it is and shifted up a byte) and its
byte weights (a texel's 2-bit index spread to a byte selects 3, 0, 2 or 1) are
restated here and compared with the plain forms; integers, exactly.
This argues the forms only: the kernels themselves are held against the
oracle on the GPU in tests/test_dxt_gpu.py."""
import numpy as np
import pytest


def u16(words):
    return np.stack([words & 0xFFFF, words >> 16], -1).reshape(len(words), -1)


@pytest.mark.parametrize("low,high", [(0, 256), (0, 2), (254, 256), (100, 101)])
def test_byte_range_of_planes(low, high):
    b = np.random.default_rng(high).integers(low, high, (4096, 16))
    w = b.reshape(-1, 4, 4)
    words = w[..., 0] | (w[..., 1] << 8) | (w[..., 2] << 16) | (w[..., 3] << 24)
    odd = u16(words)
    both = np.concatenate([odd, (odd << 8) & 0xFFFF], 1)
    assert np.array_equal(both.min(1) >> 8, b.min(1))
    assert np.array_equal(both.max(1) >> 8, b.max(1))


def test_weights_from_indices():
    for m in range(256):
        idx = (m | (m << 6) | (m << 12) | (m << 18)) & 0x03030303
        for k in range(4):
            sel = (idx >> (8 * k)) & 0xFF
            assert sel == (m >> (2 * k)) & 3
            assert (0x01020003 >> (8 * sel)) & 0xFF == (0x1203 >> (4 * sel)) & 15 == [3, 0, 2, 1][sel]
