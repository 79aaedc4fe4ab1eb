"""Products at values that ordinary data does not have: rows of zeros, very
large values, infinities and values far below the rest of their row. Against
float64, or what fp32 products and sums give."""
import numpy as np
import pytest

from tinyoai_amd import weights as W

pytestmark = pytest.mark.gpu

KQUANTS = (W.Q5_1, W.Q4_K, W.Q5_K, W.Q6_K)


def _zero_tensor(fmt, rows, cols):
    """Blocks whose constants are large (d = 40) and whose every value is zero."""
    d = np.array([40.0], np.float16).view(np.uint8)
    if fmt == W.Q5_1:
        b = np.zeros((rows * cols // 32, 24), np.uint8)
        b[:, :2] = d
    elif fmt == W.Q6_K:  # quants of 32, the middle
        b = np.zeros((rows * cols // 256, 210), np.uint8)
        b[:, 128:192], b[:, 192:208], b[:, 208:210] = 0xAA, 100, d
    else:  # quants and minima of 0
        b = np.zeros((rows * cols // 256, 144 if fmt == W.Q4_K else 176), np.uint8)
        b[:, :2], b[:, 4:8] = d, 0x3f
    return W.Tensor(fmt, rows, cols, b.reshape(-1))


@pytest.mark.parametrize("n", [33, 300])
@pytest.mark.parametrize("fmt", KQUANTS)
def test_rows_of_zeros(fmt, n):
    """A 5/6-bit row whose values are all zero, whatever its blocks' constants:
    the many-row tiles decode each value and give zeros."""
    from tinyoai_amd import hip
    w = hip.Weight(_zero_tensor(fmt, 9, 512))
    assert not np.any(w.read_values(0, 9 * 512))
    got = w.mul(np.random.default_rng(n).standard_normal((n, 512)).astype(np.float32))
    w.close()
    assert not np.any(got)  # neither a NaN nor anything but zeros
