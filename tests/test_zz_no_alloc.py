"""The no-allocation product (tinyoai_weight_mul_device_noalloc) against the
allocating one (tinyoai_weight_mul_device) through the C ABI.

The two run the same kernels; only where the activations' bf16 operand
planes live differs (the library's per-GPU array instead of a buffer grown
with hipMalloc), so the outputs must be bit-identical. Each weight takes
calls in a row with shrinking inputs (the array keeps the previous call's
planes), and an input beyond the array's limit is refused before any work.

Device buffers come from the HIP runtime the library itself is linked
against (torch bundles another one, which cannot initialise the device
once this one has in the same process).
"""
import ctypes as C

import numpy as np
import pytest

from tinyoai_amd import weights as W

pytestmark = pytest.mark.gpu


class DeviceBuffers:
    """hipMalloc'd buffers of the library's own HIP runtime."""

    def __init__(self):
        from tinyoai_amd import hip
        hip.lib()  # loads libamdhip64 as the library's dependency
        self.rt = C.CDLL("libamdhip64.so.7")
        self.rt.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        self.rt.hipFree.argtypes = [C.c_void_p]
        self.rt.hipDeviceSynchronize.argtypes = []
        self.ptrs = []

    def alloc(self, nbytes):
        p = C.c_void_p()
        assert self.rt.hipMalloc(C.byref(p), nbytes) == 0
        self.ptrs.append(p.value)
        return p.value

    def upload(self, a: np.ndarray):
        p = self.alloc(a.nbytes)
        assert self.rt.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0  # host to device
        return p

    def download(self, p, shape):
        out = np.empty(shape, np.float32)
        assert self.rt.hipDeviceSynchronize() == 0
        assert self.rt.hipMemcpy(out.ctypes.data, p, out.nbytes, 2) == 0  # device to host
        return out

    def close(self):
        for p in self.ptrs:
            self.rt.hipFree(p)
        self.ptrs = []


@pytest.mark.parametrize("dtype,rows,cols", [(W.Q8_0, 1000, 2560), (W.BF16, 512, 1024), (W.Q4_K, 300, 512)])
def test_no_alloc_product_matches_allocating_entry_point(dtype, rows, cols):
    from tinyoai_amd import hip
    rng = np.random.default_rng(rows + cols)
    if dtype == W.Q8_0:
        t = W.synthetic_q8_0(rows, cols, rng)
    elif dtype == W.BF16:
        t = W.synthetic_bf16(rows, cols, rng)
    else:
        t = W.synthetic_kquant(dtype, rows, cols, rng)
    buf = DeviceBuffers()
    w = hip.Weight(t)
    try:
        for n in (96, 17, 1):
            x = buf.upload(rng.standard_normal((n, cols)).astype(np.float32))
            y1 = buf.upload(np.zeros((n, rows), np.float32))
            y2 = buf.upload(np.full((n, rows), np.nan, np.float32))
            w.mul_device(x, n, y1)
            w.mul_device_noalloc(x, n, y2)
            a, b = buf.download(y1, (n, rows)), buf.download(y2, (n, rows))
            assert np.array_equal(a, b), (dtype, n)
            assert np.all(np.isfinite(b))
        limit = (4 << 20) // cols
        with pytest.raises(hip.TinyoaiError, match="no-allocation limit"):
            w.mul_device_noalloc(x, limit + 1, y1)
    finally:
        w.close()
        buf.close()


def test_no_alloc_calls_on_two_weights_are_ordered():
    """Calls with a null stream on two weights, back to back, each on a
    weight whose own stream would let them overlap: both results equal the
    allocating entry point's (the library runs such calls one after
    another on its own stream, so the second does not overwrite the
    first's operand planes or partials while that one still reads them)."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(77)
    t1, t2 = W.synthetic_q8_0(2048, 2560, rng), W.synthetic_bf16(1536, 2560, rng)
    buf = DeviceBuffers()
    w1, w2 = hip.Weight(t1), hip.Weight(t2)
    try:
        n = 128
        x1 = buf.upload(rng.standard_normal((n, 2560)).astype(np.float32))
        x2 = buf.upload(rng.standard_normal((n, 2560)).astype(np.float32))
        r1, r2 = buf.upload(np.zeros((n, 2048), np.float32)), buf.upload(np.zeros((n, 1536), np.float32))
        w1.mul_device(x1, n, r1)
        w2.mul_device(x2, n, r2)
        want1, want2 = buf.download(r1, (n, 2048)), buf.download(r2, (n, 1536))
        for _ in range(3):
            y1 = buf.upload(np.full((n, 2048), np.nan, np.float32))
            y2 = buf.upload(np.full((n, 1536), np.nan, np.float32))
            w1.mul_device_noalloc(x1, n, y1)
            w2.mul_device_noalloc(x2, n, y2)
            assert np.array_equal(buf.download(y1, (n, 2048)), want1)
            assert np.array_equal(buf.download(y2, (n, 1536)), want2)
    finally:
        w1.close()
        w2.close()
        buf.close()


@pytest.mark.parametrize("dtype,n", [(W.F16, 5), (W.F16, 80), (W.Q8_0, 20), (W.Q8_0, 80), (W.Q4_K, 9), (W.F32, 40)])
def test_captured_products(dtype, n):
    """tinyoai_weight_mul_device under stream capture, on a stream that has
    made no call (its scratch, where the product needs any, is what an eager
    call on another stream left): replays with new inputs, eager calls between
    them, against float64."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols = 300, 1280
    v = rng.standard_normal((rows, cols), dtype=np.float32) * np.float32(0.02)
    t = {W.F16: lambda: W.Tensor(W.F16, rows, cols, v.astype(np.float16).reshape(-1).view(np.uint8)),
         W.F32: lambda: W.Tensor(W.F32, rows, cols, v.reshape(-1).view(np.uint8)),
         W.Q8_0: lambda: W.synthetic_q8_0(rows, cols, rng),
         W.Q4_K: lambda: W.synthetic_kquant(W.Q4_K, rows, cols, rng)}[dtype]()
    buf = DeviceBuffers()
    rt, w = buf.rt, hip.Weight(t)
    dense = w.read_values(0, rows * cols).reshape(rows, cols).astype(np.float64)
    st, graph, ex = C.c_void_p(), C.c_void_p(), C.c_void_p()
    try:
        x = buf.upload(np.zeros((n, cols), np.float32))
        y, y2 = buf.alloc(n * rows * 4), buf.alloc(n * rows * 4)
        w.mul_device(x, n, y)  # eager, on the weight's own stream
        assert rt.hipDeviceSynchronize() == 0
        assert rt.hipStreamCreateWithFlags(C.byref(st), 1) == 0
        assert rt.hipStreamBeginCapture(st, 2) == 0  # relaxed: other threads may call the runtime
        w.mul_device(x, n, y, st.value)
        assert rt.hipStreamEndCapture(st, C.byref(graph)) == 0
        assert rt.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
        for _ in range(3):
            a = rng.standard_normal((n, cols)).astype(np.float32)
            assert rt.hipMemcpy(C.c_void_p(x), a.ctypes.data, a.nbytes, 1) == 0
            assert rt.hipGraphLaunch(ex, st) == 0 and rt.hipStreamSynchronize(st) == 0
            got = buf.download(y, (n, rows))
            w.mul_device(x, n, y2)
            eager = buf.download(y2, (n, rows))
            want, mag = a.astype(np.float64) @ dense.T, np.abs(a).astype(np.float64) @ np.abs(dense).T
            for r in (got, eager):  # 2^-16: bf16 planes of Q8_0 beyond 64 rows; the rest is closer
                assert np.all(np.abs(r - want) <= 2.0 ** -16 * mag)
    finally:
        if ex.value:
            rt.hipGraphExecDestroy(ex)
        if graph.value:
            rt.hipGraphDestroy(graph)
        if st.value:
            rt.hipStreamDestroy(st)
        w.close()
        buf.close()


def _captured(rt, w, st, calls, mode=0):
    """An executable graph of the calls (x, n, y) captured on st."""
    graph, ex = C.c_void_p(), C.c_void_p()
    assert rt.hipStreamBeginCapture(st, mode) == 0
    for x, n, y in calls:
        w.mul_device(x, n, y, st.value)
    assert rt.hipStreamEndCapture(st, C.byref(graph)) == 0
    assert rt.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    rt.hipGraphDestroy(graph)
    return ex


@pytest.mark.parametrize("dtype,n,warm", [(W.Q8_0, 48, 64), (W.Q8_0, 80, 0), (W.BF16, 7, 64), (W.F16, 90, 0),
                                          (W.F32, 33, 0), (W.Q4_K, 9, 32), (W.Q5_K, 70, 0)])
def test_captured_products_sum_as_eager_ones(dtype, n, warm):
    """A captured product needs no eager call before it (a larger one may have
    needed less scratch), in the mode that forbids every thread's allocations,
    and gives an eager call's bits; two graphs and eager calls on a third
    stream, all in flight together, do not disturb each other; and a graph
    captured after others were destroyed."""
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols = 700, 2048
    v = rng.standard_normal((rows, cols), dtype=np.float32) * np.float32(0.02)
    t = {W.F16: lambda: W.Tensor(W.F16, rows, cols, v.astype(np.float16).reshape(-1).view(np.uint8)),
         W.F32: lambda: W.Tensor(W.F32, rows, cols, v.reshape(-1).view(np.uint8)),
         W.BF16: lambda: W.synthetic_bf16(rows, cols, rng), W.Q8_0: lambda: W.synthetic_q8_0(rows, cols, rng)}
    t = t[dtype]() if dtype in t else W.synthetic_kquant(dtype, rows, cols, rng)
    buf = DeviceBuffers()
    rt, w = buf.rt, hip.Weight(t)
    streams, execs = [C.c_void_p() for _ in range(3)], []
    try:
        for st in streams:
            assert rt.hipStreamCreateWithFlags(C.byref(st), 1) == 0
        xs = [rng.standard_normal((max(n, warm), cols)).astype(np.float32) for _ in range(3)]
        x = [buf.upload(a) for a in xs]
        y = [buf.alloc(max(n, warm) * rows * 4) for _ in range(3)]
        if warm:
            w.mul_device(x[0], warm, y[0])
        execs += [_captured(rt, w, streams[i], [(x[i], n, y[i])] * 2) for i in range(2)]
        want = []
        for i in range(3):
            w.mul_device(x[i], n, y[2])
            want.append(buf.download(y[2], (n, rows)))
        mag = np.abs(xs[0][:n]).astype(np.float64) @ np.abs(w.read_values(0, rows * cols)).reshape(rows, cols).T
        assert np.any(want[0]) and np.all(np.abs(want[0]) <= mag)
        for round in range(3):
            for _ in range(10):
                for i in range(2):
                    assert rt.hipGraphLaunch(execs[i], streams[i]) == 0
                w.mul_device(x[2], n, y[2], streams[2].value)
            for i in range(3):
                assert np.array_equal(buf.download(y[i], (n, rows)), want[i]), (round, i)
            rt.hipGraphExecDestroy(execs[round & 1])
            execs[round & 1] = _captured(rt, w, streams[round & 1], [(x[round & 1], n, y[round & 1])])
    finally:
        for ex in execs:
            rt.hipGraphExecDestroy(ex)
        for st in streams:
            rt.hipStreamDestroy(st)
        w.close()
        buf.close()


@pytest.mark.parametrize("dtype,n", [(W.F16, 70), (W.Q8_0, 20)])
def test_products_in_flight_on_many_streams(dtype, n):
    """One weight's products in flight on twelve streams (four of them share a
    buffer) and on two threads' hipStreamPerThread, sizes growing: every output
    is that of a call alone."""
    import threading

    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols = 900, 1536
    v = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float16)
    t = W.synthetic_q8_0(rows, cols, rng) if dtype == W.Q8_0 else W.Tensor(W.F16, rows, cols, v.reshape(-1).view(np.uint8))
    buf = DeviceBuffers()
    rt, w = buf.rt, hip.Weight(t)
    streams = [C.c_void_p() for _ in range(12)]
    try:
        for st in streams:
            assert rt.hipStreamCreateWithFlags(C.byref(st), 1) == 0
        sizes = [n + 3 * i for i in range(4)]
        x = [buf.upload(rng.standard_normal((sizes[-1], cols)).astype(np.float32)) for _ in range(14)]
        y = [[buf.alloc(m * rows * 4) for m in sizes] for _ in range(14)]
        ref = buf.alloc(sizes[-1] * rows * 4)
        want = []
        for i in range(14):
            want.append([])
            for m in sizes:
                w.mul_device(x[i], m, ref)
                want[i].append(buf.download(ref, (m, rows)))
        for k, m in enumerate(sizes):
            for i, st in enumerate(streams):
                w.mul_device(x[i], m, y[i][k], st.value)

        def on_thread(i):
            rt.hipSetDevice(0)
            for k, m in enumerate(sizes):
                w.mul_device(x[i], m, y[i][k], 2)  # hipStreamPerThread

        threads = [threading.Thread(target=on_thread, args=(i,)) for i in (12, 13)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        for i in range(14):
            for k, m in enumerate(sizes):
                assert np.array_equal(buf.download(y[i][k], (m, rows)), want[i][k]), (i, m)
    finally:
        for st in streams:
            rt.hipStreamDestroy(st)
        w.close()
        buf.close()


@pytest.mark.parametrize("dtype,n", [(W.F16, 80), (W.F32, 40), (W.Q4_K, 9), (W.Q8_0, 20)])
def test_captured_no_alloc_product_matches_the_eager_one(dtype, n):
    from tinyoai_amd import hip
    rng = np.random.default_rng(n)
    rows, cols = 300, 1280
    t = {W.F32: W.synthetic_f32, W.Q8_0: W.synthetic_q8_0}.get(dtype)
    if dtype == W.F16:
        v = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float16)
        t = W.Tensor(W.F16, rows, cols, v.reshape(-1).view(np.uint8))
    else:
        t = t(rows, cols, rng) if t else W.synthetic_kquant(dtype, rows, cols, rng)
    buf = DeviceBuffers()
    rt, w = buf.rt, hip.Weight(t)
    st, graph, ex = C.c_void_p(), C.c_void_p(), C.c_void_p()
    try:
        x = buf.upload(rng.standard_normal((n, cols)).astype(np.float32))
        y, y2 = buf.upload(np.zeros((n, rows), np.float32)), buf.alloc(n * rows * 4)
        assert rt.hipStreamCreateWithFlags(C.byref(st), 1) == 0
        w.mul_device_noalloc(x, n, y2, st.value)
        want = buf.download(y2, (n, rows))
        assert rt.hipStreamBeginCapture(st, 0) == 0
        w.mul_device_noalloc(x, n, y, st.value)
        assert rt.hipStreamEndCapture(st, C.byref(graph)) == 0
        assert rt.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
        for _ in range(3):
            assert rt.hipGraphLaunch(ex, st) == 0 and rt.hipStreamSynchronize(st) == 0
            assert np.array_equal(buf.download(y, (n, rows)), want)
            w.mul_device(x, n, y2)
            assert np.array_equal(buf.download(y2, (n, rows)), want)
    finally:
        for handle, destroy in ((ex, rt.hipGraphExecDestroy), (graph, rt.hipGraphDestroy), (st, rt.hipStreamDestroy)):
            if handle.value:
                destroy(handle)
        w.close()
        buf.close()
