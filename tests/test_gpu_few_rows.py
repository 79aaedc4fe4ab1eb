"""Matrix-core products of 2 to 64 rows (F16, BF16, Q8_0) and of more rows
with F16, F32 and 5/6-bit weights, at the edges of their tiles, against
float64."""
import numpy as np
import pytest

from tinyoai_amd import weights as W

pytestmark = pytest.mark.gpu


def _weight(fmt, rows, cols, rng, oracle):
    """A tensor and its float64 values."""
    if fmt in (W.Q4_K, W.Q5_K, W.Q6_K, W.Q5_1):
        if fmt == W.Q5_1:
            b = rng.integers(0, 256, (rows * cols // 32, 24)).astype(np.uint8)
            b[:, :4] = (rng.standard_normal((rows * cols // 32, 2)) * [0.004, 0.06]).astype(np.float16).view(np.uint8)
            t = W.Tensor(fmt, rows, cols, b.reshape(-1))
        else:
            t = W.synthetic_kquant(fmt, rows, cols, rng)
        dense = oracle.read_values(oracle.weight(fmt, rows, cols, t.data), 0, rows * cols)
        return t, dense.reshape(rows, cols).astype(np.float64)
    if fmt == W.Q8_0:
        d = (rng.random(rows * cols // 32) * 2e-4).astype(np.float16)
        q = rng.integers(-128, 128, (rows * cols // 32, 32)).astype(np.int8)
        dense = d.astype(np.float64)[:, None] * q
        return W.Tensor(fmt, rows, cols, W.encode_q8_0(d.view(np.uint16), q)), dense.reshape(rows, cols)
    v = rng.standard_normal((rows, cols), dtype=np.float32) * np.float32(0.02)
    if fmt == W.F32:
        v.reshape(-1)[:2] = [3e4, 1e-30]
        return W.Tensor(fmt, rows, cols, v.reshape(-1).view(np.uint8)), v.astype(np.float64)
    if fmt == W.F16:
        h = v.astype(np.float16)
        h.reshape(-1)[:3] = np.float16([6e-8, 65504, -3e-5])[:h.size]  # subnormal and largest values
        return W.Tensor(fmt, rows, cols, h.reshape(-1).view(np.uint8)), h.astype(np.float64)
    bits = (v.view(np.uint32) >> 16).astype(np.uint16)
    return W.Tensor(fmt, rows, cols, bits.reshape(-1).view(np.uint8)), (bits.astype(np.uint32) << 16).view(
        np.float32).astype(np.float64)


def _check(fmt, rows, cols, n, rng, oracle):
    from tinyoai_amd import hip
    t, dense = _weight(fmt, rows, cols, rng, oracle)
    # rows of very different sizes, one of zeros
    x = rng.standard_normal((n, cols)).astype(np.float32) * np.float32(10.0) ** rng.integers(-20, 20, (n, 1)).astype(
        np.float32)
    x[n // 2] = 0
    g = hip.Weight(t)
    got = g.mul(x)
    g.close()
    x64 = x.astype(np.float64)
    want, mag = x64 @ dense.T, np.abs(x64) @ np.abs(dense).T
    # The operands' planes keep 16 bits of a value (bf16: BF16 weights, and
    # Q8_0 rows of an odd number of blocks) or at least 22 bits, and 38 of the
    # row's largest value (weights other than F16 too, and the product of
    # the two lo planes is left out); each of cols / 8 + 32 sums rounds to
    # 24 bits.
    bf16 = fmt == W.BF16 or (fmt == W.Q8_0 and cols % 64)
    rel = (2.0 ** -16 if bf16 else 3 * 2.0 ** -22) + (cols / 8 + 32) * 2.0 ** -24
    ax, aw = np.abs(x64), np.abs(dense)
    floor = 2.0 ** -38 * (ax.max(1, keepdims=True) * aw.sum(1) + ax.sum(1, keepdims=True) * aw.max(1))
    assert np.all(np.abs(got - want) <= rel * mag + floor), (fmt, rows, cols, n)


@pytest.mark.parametrize("n", [2, 3, 8, 16, 21, 31, 32, 33, 63, 64])
@pytest.mark.parametrize("fmt,rows,cols", [(W.F16, 1, 1), (W.F16, 31, 63), (W.F16, 257, 300), (W.F16, 2560, 1921),
                                           (W.BF16, 33, 32), (W.BF16, 300, 2560), (W.Q8_0, 37, 96), (W.Q8_0, 255, 64),
                                           (W.Q8_0, 256, 1088), (W.Q8_0, 2600, 6912)])
def test_few_row_products(oracle, fmt, rows, cols, n):
    _check(fmt, rows, cols, n, np.random.default_rng(rows + n), oracle)


@pytest.mark.parametrize("fmt,rows,cols,n", [
    (W.F16, 1, 64, 65), (W.F16, 223, 65, 127), (W.F16, 256, 100, 128), (W.F16, 257, 1921, 129), (W.F16, 300, 2560, 300),
    (W.F16, 7000, 96, 600), (W.F16, 40, 7, 200), (W.F32, 1, 64, 2), (W.F32, 255, 65, 33), (W.F32, 300, 1923, 257),
    (W.F32, 2560, 2560, 16), (W.Q4_K, 1, 256, 33), (W.Q4_K, 300, 2560, 129), (W.Q4_K, 6912, 512, 512),
    (W.Q5_K, 257, 768, 256), (W.Q5_K, 300, 2560, 70), (W.Q6_K, 255, 256, 257), (W.Q6_K, 2560, 2560, 40),
    (W.Q6_K, 2560, 2560, 500), (W.Q5_1, 300, 96, 64), (W.Q5_1, 257, 7552, 128)])
def test_products_of_many_rows(oracle, fmt, rows, cols, n):
    _check(fmt, rows, cols, n, np.random.default_rng(rows + n), oracle)


@pytest.mark.parametrize("n", [5, 70])
def test_f16_infinities_and_nan(n):
    """An infinity or NaN in a row of X stays in its row; one in the weights
    gives what fp32 products and sums give."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    v = rng.standard_normal((70, 130)).astype(np.float16)
    x = rng.standard_normal((n, 130)).astype(np.float32)
    x[1, 7], x[2, 9], x[3, 100] = np.inf, np.nan, -np.inf
    for bad in (False, True):
        if bad:
            v[3, 5], v[4, 6] = np.inf, np.nan
        g = hip.Weight(W.Tensor(W.F16, 70, 130, v.reshape(-1).view(np.uint8)))
        got = g.mul(x)
        g.close()
        with np.errstate(invalid="ignore"):
            want = x @ v.astype(np.float32).T
        fin = np.isfinite(want)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        assert np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
        assert np.allclose(got[fin], want[fin], rtol=0, atol=1e-4)


@pytest.mark.parametrize("mlp,attn,d,inter,hd,n", [
    (W.F16, W.F16, 264, 172, 8, 65), (W.F16, W.F16, 264, 172, 8, 300), (W.F16, W.F16, 320, 1000, 80, 129),
    (W.F32, W.F32, 264, 172, 8, 70), (W.F32, W.F32, 4104, 120, 8, 35), (W.Q4_K, W.Q6_K, 256, 768, 64, 33),
    (W.Q4_K, W.Q6_K, 512, 256, 128, 300), (W.Q6_K, W.Q4_K, 256, 768, 64, 129), (W.Q5_K, W.Q5_K, 512, 768, 8, 257),
    (W.Q6_K, W.Q6_K, 256, 512, 64, 70), (W.Q5_1, W.Q5_1, 320, 352, 80, 130), (W.Q4_K, W.F16, 512, 256, 64, 100)])
def test_layers_of_odd_sizes(oracle, mlp, attn, d, inter, hd, n):
    """Whole layers on the fp32-accurate tiles, alone and as pairs of products,
    with LayerNorm rows as planes (and past 4096 columns without): widths that
    are no multiple of a tile or a K step, against the oracle. Its fp32 sums
    and these differ by at most 1e-6 of a layer's range (four times that here)."""
    from tinyoai_amd import hip
    heads = d // hd
    config = W.validate_stablelm_config(dict(W.STABLELM_3B, hidden_size=d, intermediate_size=inter,
                                             num_attention_heads=heads, num_key_value_heads=heads, num_hidden_layers=2,
                                             vocab_size=300, max_position_embeddings=512))
    if mlp == W.Q5_1:
        rng = np.random.default_rng(n)
        tensors = {name: t if t.rows == 1 else _weight(W.Q5_1, t.rows, t.cols, rng, oracle)[0]
                   for name, t in W.synthetic_stablelm(config, W.F32, seed=d + n).items()}
    else:
        tensors = W.synthetic_stablelm(config, mlp, seed=d + n, attn_dtype=attn)
    ids = np.random.default_rng(n).integers(0, 300, n).astype(np.int32)
    oracle.set_threads(8)
    ref = oracle.StableLM(config, tensors, capacity=512)
    ref.trace(True)
    f = hip.StableLMForwarder(config, tensors)
    f.trace(True)
    want, got = ref.prefill(ids, 0), f.forward(0, ids)
    for a, b in zip(list(ref.trace_data()) + [want], list(f.trace_read()) + [got]):
        assert np.max(np.abs(a - b)) <= 4e-6 * float(np.ptp(a)), (np.max(np.abs(a - b)), np.ptp(a))
    f.close()
