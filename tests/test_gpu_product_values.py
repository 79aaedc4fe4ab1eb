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


def _tensor(fmt, rows, cols, rng):
    if fmt in (W.Q4_K, W.Q5_K, W.Q6_K):
        return W.synthetic_kquant(fmt, rows, cols, rng)
    if fmt == W.Q5_1:
        b = rng.integers(0, 256, (rows * cols // 32, 24)).astype(np.uint8)
        b[:, :4] = (rng.standard_normal((rows * cols // 32, 2)) * [0.004, 0.06]).astype(np.float16).view(np.uint8)
        return W.Tensor(fmt, rows, cols, b.reshape(-1))
    v = rng.standard_normal((rows, cols), dtype=np.float32) * np.float32(0.02)
    return W.Tensor(fmt, rows, cols, (v.astype(np.float16) if fmt == W.F16 else v).reshape(-1).view(np.uint8))


@pytest.mark.parametrize("n", [40, 300])
@pytest.mark.parametrize("fmt", (W.F32, W.F16) + KQUANTS)
def test_rows_of_any_size(fmt, n):
    """Rows of X from 1e-35 to 1e37, whose products with small weights are
    finite fp32 numbers: the operands' factors are applied together."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    w = hip.Weight(_tensor(fmt, 70, 512, rng))
    dense = w.read_values(0, 70 * 512).reshape(70, 512).astype(np.float64)
    x = rng.standard_normal((n, 512)) * 10.0 ** rng.uniform(-35, 37, (n, 1)) / max(1, np.abs(dense).max() / 0.05)
    x[0] *= 1e37 / np.abs(x[0]).max()
    x = x.astype(np.float32)
    got = w.mul(x)
    w.close()
    x64 = x.astype(np.float64)
    want, mag = x64 @ dense.T, np.abs(x64) @ np.abs(dense).T
    assert np.abs(want).max() > 1e36 and np.abs(want).max() < 3e38
    # 22 bits of each operand and 96 sums of 24; a total below 2^-126 in steps of 2^-149
    assert np.all(np.abs(got - want) <= (3 * 2.0 ** -22 + 96 * 2.0 ** -24) * mag + 2.0 ** -148)
