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
    if fmt == W.Q8_0:
        return W.synthetic_q8_0(rows, cols, rng)
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


def _same_kind(got, want):
    """NaN where want is, infinities where want has them and of their sign."""
    return (np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)) and
            np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)])))


@pytest.mark.parametrize("fmt,n", [(W.F32, 5), (W.F32, 300)] + [(f, n) for f in KQUANTS + (W.F16,) for n in (40, 300)])
def test_infinite_rows(fmt, n):
    """An infinity or NaN in a row of X gives what fp32 products and sums give,
    and leaves the other rows alone: with a column of weights that are zero
    (F32, F16), with weights of both signs, and beside another infinity."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols = 300, 768
    t = _tensor(fmt, rows, cols, rng)
    if fmt in (W.F32, W.F16):
        t.data.view(np.float32 if fmt == W.F32 else np.float16).reshape(rows, cols)[:, 11] = 0
    w = hip.Weight(t)
    dense = w.read_values(0, rows * cols).reshape(rows, cols).astype(np.float64)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    want = x.astype(np.float64) @ dense.T
    x[0, 7], x[1, 600], x[2, 11], x[3, 9] = np.inf, -np.inf, np.inf, np.nan
    x[4, 70], x[4, 71] = np.inf, -np.inf
    x[n - 1, cols - 1], x[n - 1, 0] = -np.inf, 3e38
    got = w.mul(x)
    w.close()
    special = [0, 1, 2, 3, 4, n - 1]
    with np.errstate(invalid="ignore", over="ignore"):
        for r in special:
            want[r] = (x[r].astype(np.float64) * dense).sum(1)
            assert _same_kind(got[r], want[r]), r
    rest = np.setdiff1d(np.arange(n), special)
    mag = np.abs(x[rest].astype(np.float64)) @ np.abs(dense).T
    assert np.all(np.abs(got[rest] - want[rest]) <= (3 * 2.0 ** -22 + 128 * 2.0 ** -24) * mag)


@pytest.mark.parametrize("fmt,n", [(W.F32, 3), (W.F32, 70), (W.F32, 257), (W.F16, 65), (W.F16, 300), (W.Q6_K, 40),
                                   (W.Q6_K, 300)] + [(f, n) for f in (W.F16, W.Q8_0) for n in (2, 5, 17, 33, 64)])
def test_values_beside_an_outlier(fmt, n):
    """Rows of X with values up to 1e60 times the rest, where every weight
    is zero, keep the precision of the rest (the bound has no term of the
    row's largest value); rows of every size at once too, and only some rows
    of a tile."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols, col = 300, 1024, 9
    t = _tensor(fmt, rows, cols, rng)
    if fmt == W.Q6_K:  # quant 32: value 0
        b = t.data.reshape(-1, 210)
        b[:, col] &= 0xF0
        b[:, 128 + col] = (b[:, 128 + col] & 0xFC) | 2
    elif fmt == W.Q8_0:
        t.data.reshape(-1, 34)[::8, 2 + col] = 0
    else:
        t.data.view(np.float32 if fmt == W.F32 else np.float16).reshape(rows, cols)[:, col::256] = 0
    w = hip.Weight(t)
    dense = w.read_values(0, rows * cols).reshape(rows, cols).astype(np.float64)
    assert not np.any(dense[:, col::256])
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[:, col::256] = 10.0 ** rng.uniform(0, 20, (n, 1))
    x[::3, col::256] = 0
    x[0] *= 1e-25
    x[0, col::256] = 1e35  # the rest is 2^-199 of it
    x[1] *= 10.0 ** rng.uniform(-15, 15, cols).astype(np.float32)
    got = w.mul(x)
    w.close()
    x64 = x.astype(np.float64)
    want, mag = x64 @ dense.T, np.abs(x64) @ np.abs(dense).T
    err = np.abs(got - want)
    ordinary = np.arange(n) != 1
    # values of at least 2^-16 of the largest hold 22 bits; the rest of a row
    # that is not marked err by 2^-39 of the largest, where most are larger
    # than 2^-16 of it: 2^-22 of their mean (Q8_0: 16 bits and 2^-22)
    assert np.all(err[ordinary] <= (4 * 2.0 ** (-16 if fmt == W.Q8_0 else -22) + 160 * 2.0 ** -24) * mag[ordinary])
    assert np.all(err[1] <= (4 if fmt == W.Q8_0 and n > 2 else 1) * 2.0 ** -22 * mag[1])


@pytest.mark.parametrize("n", [40, 300])
@pytest.mark.parametrize("fmt", (W.F32,) + KQUANTS)
def test_weights_beside_an_outlier(fmt, n):
    """Weights of up to 2^36 times the rest, in some rows' last block, where X
    is zero: the rest of the matrix keeps its precision (the bound has no term
    of the row's largest weight)."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols = 300, 1024
    t = _tensor(fmt, rows, cols, rng)
    big = slice(rows // 3, None)
    if fmt == W.F32:
        t.data.view(np.float32).reshape(rows, cols)[big, -1] = 2.0 ** 30
    else:
        per, size = W.BLOCKS[fmt]
        b = t.data.reshape(rows, cols // per, size)
        at = {W.Q5_1: [0, 2], W.Q4_K: [0, 2], W.Q5_K: [0, 2], W.Q6_K: [208]}[fmt]
        for o in at:  # block scales and minima
            b[:, :-1, o:o + 2] = np.float16(2.0 ** -20).reshape(1).view(np.uint8)
            b[big, -1, o:o + 2] = np.float16(2.0 ** 15).reshape(1).view(np.uint8)
    w = hip.Weight(t)
    dense = w.read_values(0, rows * cols).reshape(rows, cols).astype(np.float64)
    zero = 1 if fmt == W.F32 else W.BLOCKS[fmt][0]
    rest = dense[:, :-zero]
    assert np.abs(dense[big]).max() > 2.0 ** 22 * np.abs(rest).max()
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[:, cols - zero:] = 0
    got = w.mul(x)
    w.close()
    x64 = x.astype(np.float64)
    want, mag = x64 @ dense.T, np.abs(x64) @ np.abs(dense).T
    assert np.all(np.abs(got - want) <= (3 * 2.0 ** -22 + 160 * 2.0 ** -24) * mag)


@pytest.mark.parametrize("attn,mlp", [(W.F16, W.F16), (W.Q6_K, W.Q4_K)])
def test_layer_norm_with_an_outlier(attn, mlp):
    """A LayerNorm whose output has one value of 1e12 beside ordinary ones, at
    a column where the matrices that take it are zero: the logits are those of
    the same model with an ordinary value there."""
    from tinyoai_amd import hip
    config = W.validate_stablelm_config(dict(W.STABLELM_3B, hidden_size=256, intermediate_size=512, num_attention_heads=4,
                                             num_key_value_heads=4, num_hidden_layers=2, vocab_size=256,
                                             max_position_embeddings=512))
    ids = np.random.default_rng(1).integers(0, 256, 100).astype(np.int32)
    got = []
    for size in (1.0, 1e12):
        tensors = W.synthetic_stablelm(config, mlp, seed=5, attn_dtype=attn)
        for name, t in tensors.items():
            if "input_layernorm" in name:
                v = t.data.view(np.float32)
                v[9] = size if name.endswith("weight") else 0
            elif any(k in name for k in ("q_proj", "k_proj", "v_proj", "gate_proj", "up_proj")):
                if t.dtype == W.F16:
                    t.data.view(np.float16).reshape(-1, 256)[:, 9] = 0
                elif t.dtype == W.Q6_K:
                    b = t.data.reshape(-1, 210)
                    b[:, 9] &= 0xF0
                    b[:, 137] = (b[:, 137] & 0xFC) | 2
                else:  # Q4_K: the sub-block's minimum and the quant are zero
                    b = t.data.reshape(-1, 144)
                    b[:, 8] &= 0xC0
                    b[:, 16 + 9] &= 0xF0
        f = hip.StableLMForwarder(config, tensors)
        got.append(f.forward(0, ids))
        f.close()
    assert np.all(np.isfinite(got[0])) and np.std(got[0]) > 0
    assert np.max(np.abs(got[0] - got[1])) <= 1e-5 * np.max(np.abs(got[0]))


@pytest.mark.parametrize("fmt,rows,cols,n", [(W.F32, 96, 65536, 70), (W.F32, 64, 16385, 300), (W.F16, 96, 65536, 70),
                                             (W.Q6_K, 64, 65536, 200), (W.Q4_K, 64, 32768, 400)])
def test_long_rows(fmt, rows, cols, n):
    """Rows of many columns round no more than fp32 sums of 512 columns in
    float64 totals do: 512 products' chain, its error as of a random walk (in
    the norm: a quarter of sqrt(512) half-ulps of its final size, with a
    margin of a half)."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    w = hip.Weight(_tensor(fmt, rows, cols, rng))
    dense = w.read_values(0, rows * cols).reshape(rows, cols).astype(np.float64)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    got = w.mul(x)
    w.close()
    want = x.astype(np.float64) @ dense.T
    bound = 1.5 * 0.25 * np.sqrt(512.0) * 2.0 ** -24
    assert np.linalg.norm(got - want) <= bound * np.linalg.norm(want)


@pytest.mark.parametrize("n", [2, 5])
def test_long_rows_of_few(n):
    """The same of the few-row F16 product, where the matrix alone fills the
    device and each block takes its rows' whole length."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols = 65536, 4096
    v = rng.integers(0, 65536, rows * cols, dtype=np.uint16)
    v &= 0x8FFF  # sign, two exponents bits and the mantissa
    v += 0x2000
    w = hip.Weight(W.Tensor(W.F16, rows, cols, v.view(np.uint8)))
    x = rng.standard_normal((n, cols)).astype(np.float32)
    got = w.mul(x)[:, ::64]
    w.close()
    want = x.astype(np.float64) @ v.reshape(rows, cols)[::64].view(np.float16).astype(np.float64).T
    bound = 1.5 * 0.25 * np.sqrt(512.0) * 2.0 ** -24
    assert np.linalg.norm(got - want) <= bound * np.linalg.norm(want)


@pytest.mark.parametrize("fmt", KQUANTS)
@pytest.mark.parametrize("cols", [256, 2560, 12288])
def test_large_values_in_one_row(fmt, cols):
    """One row times a 5/6-bit matrix, with infinities (what fp32 products and
    sums give) and values up to 1e38 whose products with small weights are
    finite, in one lane's chunk and in every one."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(cols)
    rows = 37
    w = hip.Weight(_tensor(fmt, rows, cols, rng))
    dense = w.read_values(0, rows * cols).reshape(rows, cols).astype(np.float64)
    x = rng.standard_normal((1, cols)).astype(np.float32)
    for at, value in ((7, np.inf), (cols - 1, -np.inf), (40, np.nan)):
        y = x.copy()
        y[0, at] = value
        got = w.mul(y)
        with np.errstate(invalid="ignore"):
            assert _same_kind(got[0], (y.astype(np.float64) * dense).sum(1)), (at, value)
    y = x.copy()
    y[0, [3, 4]] = np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        assert _same_kind(w.mul(y)[0], (y.astype(np.float64) * dense).sum(1))
    one = x.copy()
    one[0, cols // 2] = 3e37 / max(1.0, np.abs(dense).max())
    every = x * np.float32(3e37 / (np.abs(x[0]) * np.abs(dense)).sum(1).max())
    for y in (one, every):
        got, y64 = w.mul(y), y.astype(np.float64)
        want, mag = y64 @ dense.T, np.abs(y64) @ np.abs(dense).T
        assert np.all(np.abs(got - want) <= (cols / 64 + 64) * 2.0 ** -24 * mag)
    w.close()


@pytest.mark.parametrize("fmt,n", [(W.F16, 20), (W.F16, 50), (W.F16, 100), (W.Q8_0, 9), (W.Q8_0, 40), (W.Q6_K, 100)])
def test_down_product_with_an_outlier(fmt, n):
    """A SiLU-gate output of up to 1e8 beside ordinary ones, where the down
    matrix is zero: the down product, the second of its launch with the o
    product, takes the marked rows from their fp32 values, and the logits are
    those of the same model with an ordinary value there (to about the error
    of its fp32 sums, 1e-6 of their range)."""
    from tinyoai_amd import hip
    d, inter = 512, 768
    config = W.validate_stablelm_config(dict(W.STABLELM_3B, hidden_size=d, intermediate_size=inter, num_attention_heads=8,
                                             num_key_value_heads=8, num_hidden_layers=2, vocab_size=256,
                                             max_position_embeddings=512))
    ids = np.random.default_rng(n).integers(0, 256, n).astype(np.int32)
    got = []
    for huge in (False, True):
        tensors = W.synthetic_stablelm(config, fmt, seed=6)
        for name, t in tensors.items():
            if name.endswith("down_proj.weight"):  # column 9 of every row
                if fmt == W.F16:
                    t.data.view(np.float16).reshape(d, inter)[:, 9] = 0
                elif fmt == W.Q8_0:
                    t.data.reshape(d, inter // 32, 34)[:, 0, 2 + 9] = 0
                else:
                    b = t.data.reshape(d, inter // 256, 210)
                    b[:, 0, 9] &= 0xF0
                    b[:, 0, 137] = (b[:, 0, 137] & 0xFC) | 2
            elif huge and name.endswith("up_proj.weight"):  # row 9
                if fmt == W.F16:
                    t.data.view(np.float16).reshape(inter, d)[9] *= np.float16(30000)
                else:
                    size, at = (34, 0) if fmt == W.Q8_0 else (210, 208)
                    t.data.reshape(inter, -1, size)[9, :, at:at + 2] = np.float16(30000).reshape(1).view(np.uint8)
        f = hip.StableLMForwarder(config, tensors)
        got.append(f.forward(0, ids))
        f.close()
    assert np.all(np.isfinite(got[0])) and np.std(got[0]) > 0
    assert np.max(np.abs(got[0] - got[1])) <= 4e-6 * np.ptp(got[0]), np.max(np.abs(got[0] - got[1])) / np.ptp(got[0])
