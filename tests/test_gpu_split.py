"""The products on the bf16 matrix units (kt_split.hip) against the same sums in 64 bits.

Bound: weights are exact and every other operand is an fp32 number split exactly, so what
remains are fp32 roundings: one per product and one per addition on a sum's path, at most
a few dozen of 2^-24 each at these sizes; normwise they add as a random walk, held to 1e-6.
"""
import ctypes

import numpy as np
import pytest

from conftest import normwise_rel
from gpu_helpers import banner, same_bits, upload_quantized

pytestmark = pytest.mark.gpu
TOL = 1e-6


def _weights(oracle_lib, k, n, bits, g, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((k, n), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
    st, q = oracle_lib.quantize(w, bits, g)
    assert st == 0
    return q


def _transposed(kt, dy, qt, dx0=None):
    m, k = dy.shape[0], qt.rows
    a = kt.DeviceBuffer.from_numpy(dy)
    dx = kt.DeviceBuffer.from_numpy(np.full((m, k), np.nan, np.float32) if dx0 is None else dx0)
    kt.MatMul.multiply_by_quantized_transposed(a, qt, dx, m, accumulate=dx0 is not None)
    kt.synchronize()
    return dx.download(np.float32).reshape(m, k)


# (m, k, n, bits, g): row tiles of 32, 64 and 128, the 128 and 512 weight rows of a tile,
# steps of 64 columns with every kind of end (odd, one column past a step, fewer than a
# step), groups of one to four 32-row blocks and of 96, runs of a slice
TRANSPOSED = [
    (1, 2300, 4100, 4, 64), (32, 513, 12001, 8, 32), (33, 1000, 2999, 4, 64), (65, 1024, 1025, 8, 64),
    (128, 385, 4096, 4, 128), (129, 2048, 577, 4, 96), (200, 640, 100, 4, 32), (300, 900, 9, 4, 64),
    (130, 9000, 64, 8, 128), (257, 512, 4672, 8, 256), (96, 4096, 7001, 4, 32),
]


@pytest.mark.parametrize("m,k,n,bits,g", TRANSPOSED)
def test_transposed_against_64_bits(kt, oracle_lib, m, k, n, bits, g):
    banner("split-transposed", m, k, n, bits, g)
    q = _weights(oracle_lib, k, n, bits, g, m + k + n)
    qt = upload_quantized(kt, q)
    rng = np.random.default_rng(m)
    dy = (rng.standard_normal((m, n)) * np.exp(4 * rng.standard_normal((m, 1)))).astype(np.float32)
    want = dy.astype(np.float64) @ q.dequantize().astype(np.float64).T
    got = _transposed(kt, dy, qt)
    # every row by itself: rows differ in size by orders of magnitude
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    print(f"  largest row error {err.max():.2e}", flush=True)
    assert err.max() <= TOL
    dx0 = rng.standard_normal((m, k)).astype(np.float32)
    assert normwise_rel(_transposed(kt, dy, qt, dx0), want + dx0) <= TOL
    assert same_bits(got, _transposed(kt, dy, qt))


# (m, k, n, bits, g, zeros): widths that are not whole quads, row tiles of 32, 64 and 128,
# column tiles that end in a byte column, steps of 64 k with every kind of end, both scale
# steps, INT8 with and without zero points
FORWARD = [
    (37, 1000, 2999, 4, 64, True), (1, 4096, 1023, 4, 32, True), (2, 4100, 2050, 8, 64, False),
    (32, 65, 65, 8, 32, True), (33, 63, 515, 8, 64, False), (64, 700, 130, 8, 96, True), (65, 2048, 257, 4, 128, True),
    (129, 577, 1030, 4, 64, True), (300, 130, 9, 4, 32, True), (150, 9000, 131, 8, 128, False), (16, 14336, 333, 4, 64, True),
]


@pytest.mark.parametrize("m,k,n,bits,g,zeros", FORWARD)
def test_forward_against_64_bits(kt, oracle_lib, m, k, n, bits, g, zeros):
    banner("split-forward", m, k, n, bits, g, zeros)
    q = _weights(oracle_lib, k, n, bits, g, m + k + n)
    rng = np.random.default_rng(m)
    if bits == 8 and zeros:
        q.zeros = rng.integers(-128, 128, q.scales.shape).astype(np.int8)
    qt = upload_quantized(kt, q)
    x = (rng.standard_normal((m, k)) * np.exp(4 * rng.standard_normal((m, 1)))).astype(np.float32)
    w = q.dequantize().astype(np.float64)
    want = x.astype(np.float64) @ w

    def product(c0=None, alpha=1.0):
        a = kt.DeviceBuffer.from_numpy(x)
        c = kt.DeviceBuffer.from_numpy(np.full((m, n), np.nan, np.float32) if c0 is None else c0)
        kt.MatMul.multiply_quantized(a, qt, c, m, accumulate=c0 is not None, alpha=alpha)
        kt.synchronize()
        return c.download(np.float32).reshape(m, n)

    got = product()
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    print(f"  largest row error {err.max():.2e}", flush=True)
    assert err.max() <= TOL
    c0 = rng.standard_normal((m, n)).astype(np.float32)
    assert normwise_rel(product(c0, -0.5), c0 - 0.5 * want) <= TOL
    assert same_bits(got, product())


def test_forward_infinities_and_nans(kt, oracle_lib):
    """An infinite or NaN input reaches its row alone, whose outputs are those of the group
    sums scale (sum a raw - zero sum a): none finite (a NaN where zero sum a is one)."""
    m, k, n = 40, 700, 333
    banner("split-forward-inf")
    for bits in (4, 8):
        q = _weights(oracle_lib, k, n, bits, 64, 15)
        qt = upload_quantized(kt, q)
        x = np.random.default_rng(16).standard_normal((m, k)).astype(np.float32)

        def product(v):
            a, c = kt.DeviceBuffer.from_numpy(v), kt.DeviceBuffer(m * n * 4)
            kt.MatMul.multiply_quantized(a, qt, c, m, accumulate=False)
            kt.synchronize()
            return c.download(np.float32).reshape(m, n)

        plain, odd = product(x), x.copy()
        odd[3, 17], odd[20, 699], odd[21, 500] = np.inf, -np.inf, np.nan
        got = product(odd)
        rest = np.setdiff1d(np.arange(m), [3, 20, 21])
        assert same_bits(got[rest], plain[rest])
        assert np.isnan(got[21]).all() and not np.isfinite(got[[3, 20]]).any()


def test_transposed_infinities_and_nans(kt, oracle_lib):
    """An infinite or NaN dY element reaches its row alone, with the products' signs; finite
    elements next to it, also the largest fp32 numbers, stay exact."""
    m, k, n = 70, 700, 2001
    banner("split-transposed-inf")
    q = _weights(oracle_lib, k, n, 4, 64, 5)
    qt = upload_quantized(kt, q)
    dy = np.random.default_rng(6).standard_normal((m, n)).astype(np.float32)
    plain = _transposed(kt, dy, qt)
    w = q.dequantize()
    odd = dy.copy()
    odd[3, 17], odd[40, 2000], odd[41, 1000] = np.inf, -np.inf, np.nan
    odd[50] = 0.0
    odd[50, 1024] = 3.4e38
    got = _transposed(kt, odd, qt)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(got[3], np.float32(np.inf) * w[:, 17], equal_nan=True)
        assert np.array_equal(got[40], np.float32(-np.inf) * w[:, 2000], equal_nan=True)
    assert np.isnan(got[41]).all()
    np.testing.assert_allclose(got[50], np.float32(3.4e38) * w[:, 1024], rtol=3e-7)
    rest = np.setdiff1d(np.arange(m), [3, 40, 41, 50])
    assert same_bits(got[rest], plain[rest])


def test_transposed_recorded_without_workspace(kt, oracle_lib):
    """Recorded on a stream that never ran eagerly (the graph has scratch of its own): replays
    equal the 64-bit result, with eager calls in between."""
    from kotensor_amd import _lib
    m, k, n = 64, 1024, 2000
    q = _weights(oracle_lib, k, n, 4, 64, 9)
    qt = upload_quantized(kt, q)
    dy = np.random.default_rng(10).standard_normal((m, n)).astype(np.float32)
    want = dy.astype(np.float64) @ q.dequantize().astype(np.float64).T
    a, dx = kt.DeviceBuffer.from_numpy(dy), kt.DeviceBuffer(m * k * 4)
    stream, graph = kt.Stream.create(), ctypes.c_void_p()
    kt.synchronize()
    banner("split-transposed-record")
    _lib.call("kt_graph_begin", stream.handle)
    try:
        kt.MatMul.multiply_by_quantized_transposed(a, qt, dx, m, accumulate=False, stream=stream)
    finally:
        _lib.call("kt_graph_end", stream.handle, ctypes.byref(graph))
    try:
        for _ in range(3):
            dx.fill_zero()
            kt.synchronize()
            _lib.call("kt_graph_launch", graph, stream.handle)
            stream.synchronize()
            assert normwise_rel(dx.download(np.float32).reshape(m, k), want) <= TOL
            assert normwise_rel(_transposed(kt, dy, qt), want) <= TOL
    finally:
        stream.synchronize()
        _lib.call("kt_graph_destroy", graph)
        stream.destroy()


def test_two_threads_on_one_stream(kt, oracle_lib):
    """Two threads call the sliced products on the null stream at once: the slices' area
    belongs to one enqueuing call at a time (the other waits for its launches)."""
    import threading

    operands = []
    for i, (m, k, n) in enumerate([(5, 4096, 1023), (40, 3000, 515)]):
        q = _weights(oracle_lib, k, n, 4, 64, 40 + i)
        rng = np.random.default_rng(50 + i)
        x, dy = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
        w = q.dequantize().astype(np.float64)
        operands.append((x, dy, upload_quantized(kt, q), x @ w, dy @ w.T))
    errors = [[], []]

    def work(i):
        x, dy, qt, y, dx = operands[i]
        m, (k, n) = x.shape[0], qt.shape
        a, b = kt.DeviceBuffer.from_numpy(x), kt.DeviceBuffer.from_numpy(dy)
        outs = [(kt.DeviceBuffer(m * n * 4), kt.DeviceBuffer(m * k * 4)) for _ in range(40)]
        for c, d in outs:
            kt.MatMul.multiply_quantized(a, qt, c, m, accumulate=False)
            kt.MatMul.multiply_by_quantized_transposed(b, qt, d, m, accumulate=False)
        kt.synchronize()
        for c, d in outs:
            errors[i] += [normwise_rel(c.download(np.float32).reshape(m, n), y), normwise_rel(d.download(np.float32).reshape(m, k), dx)]

    banner("split-two-threads")
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(len(e) == 80 and max(e) <= TOL for e in errors)


@pytest.mark.parametrize("bits,m,k,n", [(4, 40, 700, 2001), (8, 70, 1024, 1500), (4, 3, 2300, 4096)])
def test_transposed_of_rows_without_numbers(kt, oracle_lib, bits, m, k, n):
    """Many infinite and NaN dY elements: a NaN anywhere in a row makes all of its outputs
    NaNs; a row with one infinity has its products' signs; a row of infinities of both signs
    has NaNs where both meet; the other rows keep their bits."""
    banner("split-transposed-rows", bits, m, k, n)
    q = _weights(oracle_lib, k, n, bits, 64, m)
    qt, w = upload_quantized(kt, q), q.dequantize()
    dy = np.random.default_rng(m).standard_normal((m, n)).astype(np.float32)
    plain = _transposed(kt, dy, qt)
    odd = dy.copy()
    odd[0, ::7] = np.nan
    odd[1, n - 1] = -np.inf
    if m > 3:
        odd[m - 1] = np.inf
        odd[m // 2:m // 2 + 4, n // 2] = np.nan
    got = _transposed(kt, odd, qt)
    assert np.isnan(got[0]).all()
    with np.errstate(invalid="ignore"):
        assert np.array_equal(got[1], np.float32(-np.inf) * w[:, n - 1], equal_nan=True)
        changed = [0, 1]
        if m > 3:
            assert np.array_equal(got[m - 1], (np.float32(np.inf) * w).sum(1), equal_nan=True)
            assert np.isnan(got[m // 2:m // 2 + 4]).all()
            changed += [m - 1, *range(m // 2, m // 2 + 4)]
    rest = np.setdiff1d(np.arange(m), changed)
    assert same_bits(got[rest], plain[rest])


def test_rows_without_numbers_take_little_longer(kt, oracle_lib):
    """A whole input of NaNs or infinities is not summed element by element over all of K or
    N: at most 15 times the ordinary call's time (measured 2.1 and 5.6 times for the product,
    2.0 for the transposed one; with every element's whole sum the product took 167)."""
    import time
    banner("split-not-numbers-time")
    m, k, n = 512, 2048, 8191

    def seconds(x, run):
        a, out = kt.DeviceBuffer.from_numpy(x), kt.DeviceBuffer(4 * m * max(k, n))
        best = 1e9
        for _ in range(4):
            kt.synchronize()
            t = time.perf_counter()
            for _ in range(5):
                run(a, out)
            kt.synchronize()
            best = min(best, time.perf_counter() - t)
        return best

    q = _weights(oracle_lib, k, n, 4, 64, 1)
    qt = upload_quantized(kt, q)
    rng = np.random.default_rng(2)
    forward = lambda a, c: kt.MatMul.multiply_quantized(a, qt, c, m, accumulate=False)  # noqa: E731
    x = rng.standard_normal((m, k)).astype(np.float32)
    plain = seconds(x, forward)
    for v in (np.nan, np.inf):
        odd = x.copy()
        odd[:, k // 2] = v
        assert seconds(odd, forward) <= 15 * plain
    back = lambda a, c: kt.MatMul.multiply_by_quantized_transposed(a, qt, c, m, accumulate=False)  # noqa: E731
    dy = rng.standard_normal((m, n)).astype(np.float32)
    plain = seconds(dy, back)
    odd = dy.copy()
    odd[:, n // 2] = np.nan
    assert seconds(odd, back) <= 15 * plain


# both sides of where generic_matmul's short sums end: K at each number of rows, K times its waves
@pytest.mark.parametrize("m,k,n,bits,g,generic", [
    (17, 88, 257, 4, 64, True), (17, 89, 257, 4, 64, False), (16, 80, 70, 8, 32, True), (16, 81, 70, 8, 32, False),
    (4, 72, 999, 4, 64, True), (4, 73, 999, 4, 64, False), (410, 64, 1001, 4, 32, True), (411, 64, 1001, 4, 32, False),
    (33, 97, 65, 8, 32, False), (65, 95, 515, 8, 64, False),
])
def test_forward_where_short_sums_end(kt, oracle_lib, m, k, n, bits, g, generic):
    """generic_matmul adds up to 88 products a row's group, sum a q - zero sum a: a walk of
    nine roundings of 2^-24, which the difference enlarges up to four times: 2.2e-6."""
    banner("split-forward-short", m, k, n, bits, g)
    q = _weights(oracle_lib, k, n, bits, g, m + k + n)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    a, c = kt.DeviceBuffer.from_numpy(x), kt.DeviceBuffer(m * n * 4)
    kt.MatMul.multiply_quantized(a, upload_quantized(kt, q), c, m, accumulate=False)
    kt.synchronize()
    got, want = c.download(np.float32).reshape(m, n), x.astype(np.float64) @ q.dequantize().astype(np.float64)
    err = (np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)).max()
    print(f"  largest row error {err:.2e}", flush=True)
    assert err <= (2.2e-6 if generic else TOL)


def test_short_sums_of_more_rows(kt, oracle_lib):
    """64 -> 70: 17 rows take what 16 do (one launch of generic_matmul, 9.5 us; 13.4 in this
    file's kernel), with a quarter for the clock."""
    import time
    banner("split-short-sums-time")
    q = upload_quantized(kt, _weights(oracle_lib, 64, 70, 4, 64, 3))
    a, c = kt.DeviceBuffer.from_numpy(np.ones((17, 64), np.float32)), kt.DeviceBuffer(17 * 70 * 4)
    best = {16: 1e9, 17: 1e9}
    for _ in range(8):
        for m in best:
            kt.synchronize()
            t = time.perf_counter()
            for _ in range(200):
                kt.MatMul.multiply_quantized(a, q, c, m, accumulate=False)
            kt.synchronize()
            best[m] = min(best[m], time.perf_counter() - t)
    assert best[17] <= 1.25 * best[16]
