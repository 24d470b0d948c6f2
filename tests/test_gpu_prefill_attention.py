"""The prefill attention and the one-token attention of short contexts (kt_decoder.hip)
against 64 bits. Prefill: blocks of query rows that end inside a token's heads, key tiles
with every kind of end, a wave without keys of its own, both orders of the blocks, both head
dimensions; and rows with infinities.

Bound: the six products of parts per element leave out at most an fp32 rounding (2^-24 of the
product, as often above as below); with the fp32 sums of up to 1600 keys and the exponential's rounding the result is held to 1e-6 normwise."""
import numpy as np
import pytest

from conftest import normwise_rel
from gpu_helpers import banner

pytestmark = pytest.mark.gpu


def _call(kt, q, keys, values, start, heads):
    from kotensor_amd import _lib
    kvh, max_seq, d = keys.shape
    tokens = q.shape[0]
    dq, dk, dv = (kt.DeviceBuffer.from_numpy(a) for a in (q, keys, values))
    pos, out = kt.DeviceBuffer.from_numpy(np.array([start], np.int32)), kt.DeviceBuffer(q.nbytes)
    _lib.call("kt_attention", dq.ptr, tokens, pos.ptr, start + tokens, dk.ptr, dv.ptr, 0, max_seq, heads, kvh, d, out.ptr, None)
    kt.synchronize()
    return out.download(np.float32).reshape(q.shape)


def _exact(q, keys, values, start, heads):
    kvh, _, d = keys.shape
    tokens = q.shape[0]
    out = np.empty(q.shape)
    visible = np.arange(start + tokens)[None] <= start + np.arange(tokens)[:, None]
    for h in range(heads):
        k, v = (a[h // (heads // kvh), :start + tokens].astype(np.float64) for a in (keys, values))
        s = q[:, h * d:(h + 1) * d].astype(np.float64) @ k.T / np.sqrt(d)
        p = np.where(visible, np.exp(s - np.where(visible, s, -np.inf).max(1, keepdims=True)), 0.0)
        out[:, h * d:(h + 1) * d] = p @ v / p.sum(1, keepdims=True)
    return out


@pytest.mark.parametrize("tokens,start,heads,kvh,d", [
    (16, 0, 4, 4, 64), (17, 47, 14, 2, 64), (64, 0, 32, 8, 64), (65, 63, 8, 1, 64), (100, 1500, 4, 1, 64),
    (700, 1, 8, 8, 64), (16, 0, 8, 8, 128), (33, 95, 16, 2, 128), (130, 200, 7, 1, 128), (40, 3, 3, 1, 64),
    (191, 0, 8, 8, 64), (160, 32, 14, 2, 64), (33, 190, 8, 1, 128), (16, 240, 9, 1, 64), (257, 0, 5, 5, 128),
])
def test_prefill_attention_against_64_bits(kt, tokens, start, heads, kvh, d):
    banner("prefill-attention", tokens, start, heads, kvh, d)
    rng = np.random.default_rng(tokens + start)
    max_seq = start + tokens + 5
    q = (2.0 * rng.standard_normal((tokens, heads * d))).astype(np.float32)
    keys, values = (rng.standard_normal((kvh, max_seq, d)).astype(np.float32) for _ in range(2))
    keys[:, start + tokens:] = np.nan  # past the last key: never used
    err = normwise_rel(_call(kt, q, keys, values, start, heads), _exact(q, keys, values, start, heads))
    print(f"  error {err:.2e}", flush=True)
    assert err <= 1e-6


def test_prefill_attention_recorded_without_workspace(kt):
    """Recorded on a stream that never ran eagerly (the graph has an area of its own for the
    parts): replays equal the 64-bit result, with eager calls in between."""
    import ctypes

    from kotensor_amd import _lib
    tokens, heads, kvh, d = 210, 8, 2, 64
    rng = np.random.default_rng(3)
    q = rng.standard_normal((tokens, heads * d)).astype(np.float32)
    keys, values = (rng.standard_normal((kvh, tokens, d)).astype(np.float32) for _ in range(2))
    want = _exact(q, keys, values, 0, heads)
    dq, dk, dv, pos = (kt.DeviceBuffer.from_numpy(a) for a in (q, keys, values, np.zeros(1, np.int32)))
    out, stream, graph = kt.DeviceBuffer(q.nbytes), kt.Stream.create(), ctypes.c_void_p()
    kt.synchronize()
    banner("prefill-attention-record")
    _lib.call("kt_graph_begin", stream.handle)
    try:
        _lib.call("kt_attention", dq.ptr, tokens, pos.ptr, tokens, dk.ptr, dv.ptr, 0, tokens, heads, kvh, d, out.ptr, stream.handle)
    finally:
        _lib.call("kt_graph_end", stream.handle, ctypes.byref(graph))
    try:
        for _ in range(3):
            out.fill_zero()
            kt.synchronize()
            _lib.call("kt_graph_launch", graph, stream.handle)
            stream.synchronize()
            assert normwise_rel(out.download(np.float32).reshape(q.shape), want) <= 1e-6
            assert normwise_rel(_call(kt, q, keys, values, 0, heads), want) <= 1e-6
    finally:
        stream.synchronize()
        _lib.call("kt_graph_destroy", graph)
        stream.destroy()


@pytest.mark.parametrize("start,heads,kvh", [(0, 32, 8), (15, 14, 2), (16, 1, 1), (255, 8, 8), (256, 32, 8), (511, 9, 1), (639, 16, 2)])
def test_one_token_of_a_short_context_against_64_bits(kt, start, heads, kvh):
    """The kernel of one workgroup per query head: a wave's rows, passes of 256 keys and the
    longest context it takes; also inside a longer cache than its keys."""
    banner("one-token-attention", start, heads, kvh)
    rng = np.random.default_rng(start)
    q = (2.0 * rng.standard_normal((1, heads * 64))).astype(np.float32)
    keys, values = (rng.standard_normal((kvh, start + 40, 64)).astype(np.float32) for _ in range(2))
    keys[:, start + 1:], values[:, start + 1:] = np.nan, np.nan  # never used
    err = normwise_rel(_call(kt, q, keys, values, start, heads), _exact(q, keys, values, start, heads))
    assert err <= 1e-6


@pytest.mark.parametrize("d,tokens", [(64, 70), (128, 70), (64, 200), (128, 200)])
def test_prefill_attention_infinities(kt, d, tokens):
    """A key whose score is minus infinity adds nothing, an infinite value makes infinities
    of the rows that see it, a NaN query NaNs of its own row; other rows keep their values."""
    heads, kvh = 4, 2
    rng = np.random.default_rng(7)
    q = rng.standard_normal((tokens, heads * d)).astype(np.float32)
    q[:, ::d] = np.abs(q[:, ::d]) + 0.1  # each head's first dim positive
    keys, values = (rng.standard_normal((kvh, tokens, d)).astype(np.float32) for _ in range(2))
    want = _exact(q, keys, values, 0, heads)
    keys[0, 5] = 0.0
    keys[0, 5, 0] = -np.inf
    values[1, 60, 3] = np.inf
    q[20, 2 * d + 1] = np.nan
    banner("prefill-attention-inf", d, tokens)
    got = _call(kt, q, keys, values, 0, heads)
    plain = keys.copy()
    plain[0, 5, 0] = -1e6  # the same weights: nothing
    ref = _exact(q, plain, np.where(np.isinf(values), 0.0, values).astype(np.float32), 0, heads)
    g0, r0 = got[:, :2 * d], ref[:, :2 * d]
    assert normwise_rel(np.delete(g0, 5, 0), np.delete(r0, 5, 0)) <= 1e-6 and np.isfinite(g0).all()
    third = got[:, 2 * d:3 * d]
    assert np.isnan(third[20]).all()
    assert np.isposinf(third[60:, 3]).all()
    keep = np.setdiff1d(np.arange(60), [20])
    assert normwise_rel(third[keep], want[keep, 2 * d:3 * d]) <= 1e-6


@pytest.mark.parametrize("d,tokens", [(64, 70), (128, 70), (64, 200), (128, 200)])
def test_prefill_attention_of_full_significands(kt, d, tokens):
    """Scores of one product 64 a * a against 64 a * 1 with a = 1 + 2^-7 - 2^-23, all of whose
    bits below the first bf16 part are set: cut into parts, not rounded, the products that are
    left out are 4.7e-7 of the score 65 (in powers of two).

    Bound: a score leaves two fp32 roundings, the largest of its sum at 65, 3.9e-6 each; the
    weight of the first keys, 2^0.5 / (1 + 2^0.5), moves by its complement times ln 2 of that:
    2.2e-6 (cut off: 8.7e-6 more)."""
    a = np.float32(1 + 2.0**-7 - 2.0**-23)
    scale = np.float32(1.0 / np.sqrt(np.float32(d))) * np.float32(1.4426950408889634)
    near = np.float32(64 * a / scale) + np.arange(-4, 5, dtype=np.float32) * np.float32(2.0**-15)
    first = near[near * scale == 64 * a]  # the kernel scales q by this
    banner("prefill-attention-significands", d, tokens, first.size)
    q, keys, values = (np.zeros(s, np.float32) for s in ((tokens, d), (1, tokens, d), (1, tokens, d)))
    q[:, 0] = first[0]
    keys[0, :, 0] = np.where(np.arange(tokens) % 2 == 0, a, np.float32(1))
    values[0, ::2] = 1.0
    err = normwise_rel(_call(kt, q, keys, values, 0, 1), _exact(q, keys, values, 0, 1))
    print(f"  error {err:.2e}", flush=True)
    assert err <= 2.2e-6


@pytest.mark.parametrize("d,tokens", [(64, 100), (128, 100), (64, 1024), (128, 300)])
def test_prefill_attention_of_rows_without_numbers(kt, d, tokens):
    """An infinite value at the third key: every later row of its heads is summed from the fp32
    values, dealt to all waves, and keeps its other dims' values; rows with a NaN query are
    left as NaNs. In at most 15 times the ordinary call's time (measured 7; 97 when one wave
    took a block's rows, lane by lane)."""
    import time
    heads, kvh = 8, 2
    rng = np.random.default_rng(tokens)
    q = rng.standard_normal((tokens, heads * d)).astype(np.float32)
    keys, values = (rng.standard_normal((kvh, tokens, d)).astype(np.float32) for _ in range(2))
    banner("prefill-attention-not-numbers", d, tokens)
    ref = _exact(q, keys, values, 0, heads)

    def seconds():
        best = 1e9
        for _ in range(3):
            from kotensor_amd import _lib
            dq, dk, dv, pos, out = *(kt.DeviceBuffer.from_numpy(a) for a in (q, keys, values, np.zeros(1, np.int32))), kt.DeviceBuffer(q.nbytes)
            kt.synchronize()
            t = time.perf_counter()
            for _ in range(5):
                _lib.call("kt_attention", dq.ptr, tokens, pos.ptr, tokens, dk.ptr, dv.ptr, 0, tokens, heads, kvh, d, out.ptr, None)
            kt.synchronize()
            best = min(best, time.perf_counter() - t)
        return best

    plain = seconds()
    values[1, 2, 5] = np.inf
    q[tokens - 1, 5 * d + 7] = np.nan
    assert seconds() <= 15 * plain
    got = _call(kt, q, keys, values, 0, heads)
    assert np.isnan(got[tokens - 1, 5 * d:6 * d]).all()
    assert normwise_rel(got[:, :4 * d], ref[:, :4 * d]) <= 1e-6  # the other key/value head
    mine, want = got[:, 4 * d:].reshape(tokens, 4, d).copy(), ref[:, 4 * d:].reshape(tokens, 4, d).copy()
    mine[tokens - 1, 1], want[tokens - 1, 1] = 0.0, 0.0
    hit = mine[2:, :, 5]
    assert np.isposinf(np.delete(hit.reshape(-1), (tokens - 3) * 4 + 1)).all()
    mine[2:, :, 5], want[2:, :, 5] = 0.0, 0.0
    assert normwise_rel(mine, want) <= 1e-6
