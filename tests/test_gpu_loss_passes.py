"""The fused cross-entropy's passes of many chunks (kt_loss.hip) against the oracle, where a
pass ends: more rows than 2^25 logits hold, a last chunk of at most 16 rows (its product on
its own), chunks of at most 16 rows, rows beyond the registers' 32768 logits, a single class.

Bound: as tests/test_gpu_loss.py, the products' 2e-3 normwise."""
import numpy as np
import pytest

import oracle
from conftest import normwise_rel
from gpu_helpers import banner, same_bits
from test_gpu_loss import TOL, _run, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n,rows,bits,g", [
    (64, 151936, 230, 4, 64),  # 27 rows a chunk, 216 a pass; the second pass has 14
    (32, 300000, 30, 8, 32),   # 13 rows a chunk
    (64, 32768, 145, 4, 32),   # 128 rows a chunk and 17 more in one product
    (64, 32769, 135, 8, 64),   # 127 rows a chunk, 8 more on their own; one logit past the registers
    (64, 1, 20, 8, 64),
])
def test_passes_match_the_oracle(kt, oracle_lib, k, n, rows, bits, g):
    banner("fused-ce-passes", k, n, rows, bits, g)
    q, head, bias, hidden, targets = _setup(kt, oracle_lib, k, n, rows, bits, g, k + n)
    loss, hg, bg = _run(kt, head, hidden, targets)
    want_loss, want_hg, want_bg = oracle.fused_cross_entropy(hidden, q, targets, bias, threads=16)
    assert abs(loss - want_loss) <= TOL * max(1.0, abs(want_loss))
    assert normwise_rel(hg, want_hg) <= TOL
    assert normwise_rel(bg, want_bg) <= TOL
    loss2, hg2, bg2 = _run(kt, head, hidden, targets)
    assert loss2 == loss and same_bits(hg, hg2) and same_bits(bg, bg2)


def test_scratch_kept_with_the_stream(kt, oracle_lib):
    """The scratch area grows and is reused between calls of different sizes on a stream, and
    a stream made after another was destroyed starts without it: always the same bits."""
    banner("fused-ce-scratch")
    q, head, bias, hidden, targets = _setup(kt, oracle_lib, 64, 2000, 40, 4, 64, 3)
    small = _run(kt, head, hidden[:3], targets[:3])
    whole = _run(kt, head, hidden, targets)
    for _ in range(2):
        stream = kt.Stream.create()
        for rows, want in ((3, small), (40, whole), (3, small)):
            h = kt.DeviceTensor.from_numpy(hidden[:rows])
            hg, bg = kt.DeviceTensor.zeros(h.shape), kt.DeviceTensor.zeros((1, head.out_size))
            kt.synchronize()  # the zeros, on the null stream
            out = kt.fused_cross_entropy_loss(h, head, targets[:rows], hidden_grad=hg, bias_grad=bg, stream=stream)
            stream.synchronize()
            assert out.item() == want[0]
            assert same_bits(out.hidden_grad.numpy(), want[1]) and same_bits(out.bias_grad.numpy().reshape(-1), want[2])
        stream.destroy()


def test_scratch_of_wide_rows(kt):
    """1024 classes of 8192 inputs: a chunk is 4096 rows, 285 MB of logits, rows and gradients,
    and a pass one chunk. Two passes take no more than one, and give the halves' gradients:
    with half the scale of one pass's, the same numbers down to fp32 rounding (the weights of
    the scale are powers of two)."""
    from test_gpu_recorded_scratch import _free_bytes
    rows, k, n = 8192, 8192, 1024
    banner("fused-ce-wide-rows")
    rng = np.random.default_rng(8)
    head = kt.QuantizedLinear(k, n, kt.Quantization(4, 64))
    head.weight = kt.QuantizedTensor.quantize((rng.standard_normal((k, n), dtype=np.float32) * np.float32(0.02)), k, n, kt.Quantization(4, 64))
    head.bias = kt.DeviceTensor.zeros((1, n))
    hidden, targets = rng.standard_normal((rows, k), dtype=np.float32), rng.integers(0, n, rows).astype(np.int32)

    def run(h, t):
        d = kt.DeviceTensor.from_numpy(h)
        hg, bg = kt.DeviceTensor.zeros(d.shape), kt.DeviceTensor.zeros((1, n))
        kt.synchronize()
        kt.release_scratch()
        before = _free_bytes()
        out = kt.fused_cross_entropy_loss(d, head, t, hidden_grad=hg, bias_grad=bg)
        taken = before - _free_bytes()
        kt.synchronize()
        return out.item(), hg.numpy(), bg.numpy(), taken

    loss, hg, bg, taken = run(hidden, targets)
    halves = [run(hidden[s], targets[s]) for s in (slice(0, 4096), slice(4096, None))]
    print(f"  {taken >> 20} MB, one chunk {halves[0][3] >> 20} MB", flush=True)
    assert taken <= 400 << 20
    assert abs(loss - 0.5 * (halves[0][0] + halves[1][0])) <= 1e-6 * loss
    assert normwise_rel(hg, 0.5 * np.concatenate([h[1] for h in halves])) <= 1e-6
    assert normwise_rel(bg, 0.5 * (halves[0][2] + halves[1][2])) <= 1e-6


def test_two_threads_on_one_stream(kt, oracle_lib):
    """Two threads' losses on the null stream, in one area one after the other: always the bits
    each has alone."""
    import threading
    banner("fused-ce-two-threads")
    cases = [_setup(kt, oracle_lib, 64, n, rows, 4, 64, n) for n, rows in ((2000, 40), (3001, 130))]
    want = [_run(kt, head, hidden, targets) for _, head, _, hidden, targets in cases]
    bad = []

    def work(i):
        _, head, _, hidden, targets = cases[i]
        for _ in range(20):
            got = _run(kt, head, hidden, targets)
            bad.append(got[0] != want[i][0] or not same_bits(got[1], want[i][1]) or not same_bits(got[2], want[i][2]))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(bad) == 40 and not any(bad)
