"""Calls with scratch of their own (split products, prompt attention on parts) recorded into
graphs: the graph has its own scratch, so replays on any stream, next to eager calls or to
other graphs' replays, give the eager call's bits."""
import contextlib
import ctypes

import numpy as np
import pytest

from gpu_helpers import banner, same_bits, upload_quantized

pytestmark = pytest.mark.gpu


class _Call:
    """One call on operands of its own: run() enqueues it, result() downloads its output."""

    def __init__(self, kt, shape):
        self.kt, self.out = kt, kt.DeviceBuffer(int(np.prod(shape)) * 4)

    def result(self):
        return self.out.download(np.float32)

    def eager(self):
        self.out.fill_zero()
        self.run(None)
        self.kt.synchronize()
        return self.result()


class _Transposed(_Call):
    def __init__(self, kt, oracle_lib, m, k, n, seed):
        super().__init__(kt, (m, k))
        rng = np.random.default_rng(seed)
        st, q = oracle_lib.quantize((rng.standard_normal((k, n)) * 0.02).astype(np.float32), 4, 64)
        assert st == 0
        self.q, self.m, self.a = upload_quantized(kt, q), m, kt.DeviceBuffer.from_numpy(rng.standard_normal((m, n)).astype(np.float32))

    def run(self, stream):
        self.kt.MatMul.multiply_by_quantized_transposed(self.a, self.q, self.out, self.m, accumulate=False, stream=stream)


class _Forward(_Call):
    def __init__(self, kt, oracle_lib, m, k, n, seed):
        super().__init__(kt, (m, n))
        rng = np.random.default_rng(seed)
        st, q = oracle_lib.quantize((rng.standard_normal((k, n)) * 0.02).astype(np.float32), 4, 64)
        assert st == 0
        self.q, self.m, self.a = upload_quantized(kt, q), m, kt.DeviceBuffer.from_numpy(rng.standard_normal((m, k)).astype(np.float32))

    def run(self, stream):
        self.kt.MatMul.multiply_quantized(self.a, self.q, self.out, self.m, accumulate=False, stream=stream)


class _Attention(_Call):
    def __init__(self, kt, oracle_lib, tokens, heads, kvh, seed):
        super().__init__(kt, (tokens, heads * 64))
        rng = np.random.default_rng(seed)
        self.shape = tokens, heads, kvh
        self.q, self.k, self.v = (kt.DeviceBuffer.from_numpy(rng.standard_normal((tokens * h * 64,)).astype(np.float32)) for h in (heads, kvh, kvh))
        self.pos = kt.DeviceBuffer.from_numpy(np.zeros(1, np.int32))

    def run(self, stream):
        from kotensor_amd import _lib
        tokens, heads, kvh = self.shape
        _lib.call("kt_attention", self.q.ptr, tokens, self.pos.ptr, tokens, self.k.ptr, self.v.ptr, 0, tokens, heads, kvh, 64, self.out.ptr,
                  stream.handle if stream else None)


# kind, sizes of the call, sizes of a larger one
KINDS = [(_Transposed, (64, 1024, 2000), (300, 2048, 4000)), (_Forward, (37, 1000, 2999), (150, 4000, 3001)), (_Attention, (210, 8, 2), (700, 16, 4))]
IDS = ["transposed", "odd width", "attention"]


def _hip():
    """The HIP runtime that the library loaded."""
    with open("/proc/self/maps") as maps:
        return ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))


@contextlib.contextmanager
def _recorded(call, stream):
    from kotensor_amd import _lib
    graph = ctypes.c_void_p()
    _lib.call("kt_graph_begin", stream.handle)
    try:
        call.run(stream)
    finally:
        _lib.call("kt_graph_end", stream.handle, ctypes.byref(graph))
    try:
        yield graph
    finally:
        call.kt.synchronize()
        _lib.call("kt_graph_destroy", graph)


def _replay(call, graph, stream):
    from kotensor_amd import _lib
    call.out.fill_zero()
    call.kt.synchronize()
    _lib.call("kt_graph_launch", graph, stream.handle)
    stream.synchronize()
    return call.result()


@pytest.mark.parametrize("kind,sizes,larger", KINDS, ids=IDS)
@pytest.mark.parametrize("eager_first", [True, False])
def test_replays_give_the_eager_bits(kt, oracle_lib, kind, sizes, larger, eager_first):
    """Recorded on a stream with and without eager calls before; a larger eager call on it
    then replaces its area, and the stream ends before the graph does."""
    banner("recorded-scratch", kind.__name__, eager_first)
    call, big = kind(kt, oracle_lib, *sizes, 1), kind(kt, oracle_lib, *larger, 2)
    want, want_big = call.eager(), big.eager()
    stream, other = kt.Stream.create(), kt.Stream.create()
    if eager_first:
        call.run(stream)
        stream.synchronize()
        assert same_bits(call.result(), want)
    with _recorded(call, stream) as graph:
        assert same_bits(_replay(call, graph, stream), want)
        big.run(stream)
        stream.synchronize()
        assert same_bits(big.result(), want_big)
        assert same_bits(_replay(call, graph, stream), want)
        stream.destroy()
        for _ in range(2):
            assert same_bits(_replay(call, graph, other), want)
            assert same_bits(big.eager(), want_big)
        other.synchronize()
    other.destroy()


@pytest.mark.parametrize("kind,sizes,larger", KINDS, ids=IDS)
def test_replays_on_other_streams_do_not_meet(kt, oracle_lib, kind, sizes, larger):
    """Two graphs recorded on one stream, replayed on two others while that stream runs a
    third call eagerly: each has the bits it has alone, every time."""
    from kotensor_amd import _lib
    banner("recorded-scratch-streams", kind.__name__)
    calls = [kind(kt, oracle_lib, *sizes, seed) for seed in (1, 2, 3)]
    want = [c.eager() for c in calls]
    streams = [kt.Stream.create() for _ in range(3)]
    calls[2].run(streams[2])
    streams[2].synchronize()
    with _recorded(calls[0], streams[2]) as a, _recorded(calls[1], streams[2]) as b:
        for _ in range(5):
            for c in calls:
                c.out.fill_zero()
            kt.synchronize()
            for _ in range(20):
                _lib.call("kt_graph_launch", a, streams[0].handle)
                _lib.call("kt_graph_launch", b, streams[1].handle)
                calls[2].run(streams[2])
            for s in streams:
                s.synchronize()
            assert all(same_bits(c.result(), w) for c, w in zip(calls, want))
    for s in streams:
        s.destroy()


@pytest.mark.parametrize("kind,sizes", [(_Transposed, (16, 1024, 4000)), (_Transposed, (200, 640, 1000)), (_Forward, (37, 1000, 2999)), (_Attention, (210, 8, 2))])
def test_a_callers_own_capture(kt, oracle_lib, kind, sizes):
    """A capture begun with HIP itself records the forms without scratch: the row-by-row
    kernel (16 rows) or one slice, the attention kernel that splits tiles itself. Their sums
    have another order: 1e-6 normwise, the bound of the products' and the attention's tests."""
    banner("recorded-scratch-own-capture", kind.__name__, *sizes)
    call = kind(kt, oracle_lib, *sizes, 4)
    want = call.eager()
    hip = _hip()
    stream, graph, exe = kt.Stream.create(), ctypes.c_void_p(), ctypes.c_void_p()
    call.run(stream)  # an area that the recorded call must not take
    stream.synchronize()
    handle = ctypes.c_void_p(stream.handle)
    assert hip.hipStreamBeginCapture(handle, 1) == 0  # thread-local
    try:
        call.run(stream)
    finally:
        assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    for _ in range(3):
        got = _replay(call, exe, stream)
        assert np.linalg.norm(got.astype(np.float64) - want) <= 1e-6 * np.linalg.norm(want)
        assert same_bits(call.eager(), want)
    assert hip.hipGraphExecDestroy(exe) == 0
    stream.destroy()


@pytest.mark.parametrize("kind,sizes,larger", KINDS, ids=IDS)
def test_a_capture_the_caller_ends(kt, oracle_lib, kind, sizes, larger):
    """Begun with kt_graph_begin and ended with HIP itself: the library does not see this
    graph's end, so its scratch stays allocated, also after the stream's next graph is gone."""
    from kotensor_amd import _lib
    banner("recorded-scratch-callers-end", kind.__name__)
    call, other = kind(kt, oracle_lib, *sizes, 6), kind(kt, oracle_lib, *larger, 7)
    want, want_other = call.eager(), other.eager()
    hip, stream = _hip(), kt.Stream.create()
    graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
    _lib.call("kt_graph_begin", stream.handle)
    try:
        call.run(stream)
    finally:
        assert hip.hipStreamEndCapture(ctypes.c_void_p(stream.handle), ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    with _recorded(other, stream) as later:
        assert same_bits(_replay(other, later, stream), want_other)
        assert same_bits(_replay(call, exe, stream), want)
    kt.release_scratch()
    for _ in range(2):
        assert same_bits(_replay(call, exe, stream), want)
        assert same_bits(other.eager(), want_other)
    assert hip.hipGraphExecDestroy(exe) == 0
    stream.destroy()


@pytest.mark.parametrize("kind,sizes,larger", KINDS, ids=IDS)
def test_two_threads_give_the_same_bits(kt, oracle_lib, kind, sizes, larger):
    """Two threads call on the null stream at once: each result has the bits it has alone."""
    import threading

    banner("scratch-two-threads", kind.__name__)
    calls = [[kind(kt, oracle_lib, *s, 10 * i + j) for j, s in enumerate((sizes, larger))] for i in range(2)]
    want = [[c.eager() for c in pair] for pair in calls]
    bad = []

    def work(i):
        for _ in range(20):
            for c in calls[i]:
                c.run(None)
        kt.synchronize()
        bad.extend(not same_bits(c.result(), w) for c, w in zip(calls[i], want[i]))

    for pair in calls:
        for c in pair:
            c.out.fill_zero()
    kt.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(bad) == 4 and not any(bad)


# slices of every size: many, few, and (2560 rows) two that would need 62.5 MiB, more than the
# fixed array's general area
@pytest.mark.parametrize("m,k,n,bits", [(1, 4096, 1023, 4), (37, 1000, 2999, 4), (200, 2000, 515, 8), (2560, 256, 3199, 4)])
def test_noalloc_gives_the_bits_of_the_plain_product(kt, oracle_lib, m, k, n, bits):
    from kotensor_amd import _lib
    banner("scratch-noalloc", m, k, n, bits)
    rng = np.random.default_rng(m)
    st, q = oracle_lib.quantize((rng.standard_normal((k, n)) * 0.02).astype(np.float32), bits, 64)
    assert st == 0
    qt, a = upload_quantized(kt, q), kt.DeviceBuffer.from_numpy(rng.standard_normal((m, k)).astype(np.float32))
    got = []
    for entry in ("kt_qmatmul", "kt_qmatmul_noalloc"):
        c = kt.DeviceBuffer(m * n * 4)
        _lib.call(entry, a.ptr, m, ctypes.byref(qt.qweight), c.ptr, 0, ctypes.c_float(1.0), None)
        kt.synchronize()
        got.append(c.download(np.float32))
    assert same_bits(*got)


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_scratch_is_given_back(kt, oracle_lib):
    """What calls kept on the null stream, on a stream of the library and on one that its
    owner destroyed, and what graphs had: free again after release_scratch and the graphs'
    ends (within 8 MiB for what the runtime itself keeps; a call here keeps 40 MB)."""
    banner("scratch-given-back")
    call = _Transposed(kt, oracle_lib, 512, 2048, 4096, 5)
    call.eager()
    kt.release_scratch()
    before = _free_bytes()
    call.eager()
    assert _free_bytes() < before - (32 << 20)
    own, theirs = kt.Stream.create(), ctypes.c_void_p()
    hip = _hip()
    assert hip.hipStreamCreate(ctypes.byref(theirs)) == 0
    for s in (own, kt.Stream(theirs.value)):
        call.run(s)
        s.synchronize()
    own.destroy()
    assert hip.hipStreamDestroy(theirs) == 0
    want = call.eager()
    stream = kt.Stream.create()
    for _ in range(10):  # 40 MB a graph
        with _recorded(call, stream) as graph:
            assert same_bits(_replay(call, graph, stream), want)
    stream.destroy()
    kt.release_scratch()
    assert _free_bytes() > before - (8 << 20)
    assert same_bits(call.eager(), want)


@pytest.mark.parametrize("kind,sizes,larger", KINDS, ids=IDS)
def test_the_per_thread_stream(kt, oracle_lib, kind, sizes, larger):
    """hipStreamPerThread is one handle for a stream of each thread: two threads' calls on it
    run at once and keep their bits."""
    import threading

    banner("scratch-per-thread-stream", kind.__name__)
    calls = [[kind(kt, oracle_lib, *s, 10 * i + j) for j, s in enumerate((sizes, larger))] for i in range(2)]
    want = [[c.eager() for c in pair] for pair in calls]
    for pair in calls:
        for c in pair:
            c.out.fill_zero()
    kt.synchronize()
    bad = []

    def work(i):
        stream = kt.Stream(2)
        for _ in range(20):
            for c in calls[i]:
                c.run(stream)
        stream.synchronize()
        bad.extend(not same_bits(c.result(), w) for c, w in zip(calls[i], want[i]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(bad) == 4 and not any(bad)
