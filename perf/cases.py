"""Performance cases of kotensor_amd: the calls a program that uses this library makes,
through its public entry points, with the work each cannot do without, the tolerance two
correct implementations agree within, and a 64-bit restatement of each result.

``listed()`` are fixed sizes; ``draw(rng)`` gives further cases of the same ranges. A
case's "kind" selects the call:

* linear:    QuantizedLinear forwards of 1 to 3 projections that share their input (q/k/v,
             gate/up, down, head), for 1 row (a decode step) to 2048 rows (a prompt);
* quantize:  kt_quantize of an fp32 weight into the caller's buffers (model import);
* backward:  the input gradient dX = dY . deq(W)^T (adapter training);
* loss:      the fused projection + cross-entropy with its gradients (training);
* attention: the cached attention of one layer, a decode step (with RoPE and the cache
             append) or a prompt;
* request:   a whole decoder: a prompt's prefill, then decode steps as graph replays.
"""
import ctypes
import math

import numpy as np
import torch

import kotensor_amd as kt
from kotensor_amd import _lib


# ---- the cases ------------------------------------------------------------------------

def _linear(name, m, k, outs, bits, group, packed=True):
    return {"name": name, "kind": "linear", "m": m, "k": k, "outs": outs, "bits": bits, "group": group, "packed": packed}


def listed():
    return [
        # the smallest call: q/k/v of a 0.5B decoder's decode step (896 -> 896, 128, 128)
        _linear("qkv_step", 1, 896, "896,128,128", 4, 64),
        # an 8B decoder's gate projection in a decode step: the weight stream alone
        _linear("gate_step", 1, 4096, "14336", 4, 64),
        # the same with eight sequences decoded together
        _linear("gate_batch8", 8, 4096, "14336", 4, 64),
        # the 8B down projection for 64 rows (a large decode batch, a short prompt)
        _linear("down_batch64", 64, 14336, "4096", 4, 64),
        # gate and up of a 1B decoder over a 512-token prompt, INT8
        _linear("gateup_prompt", 512, 2048, "8192,8192", 8, 32),
        # odd rows, inputs and outputs, no device copy of the weight (an unprepared layer)
        _linear("odd_linear", 37, 1000, "2999", 4, 64, False),
        # importing an 8B decoder: one gate projection quantized
        {"name": "quantize_gate", "kind": "quantize", "k": 4096, "n": 14336, "bits": 4, "group": 64},
        # adapter training on a 1B decoder: the input gradient of a gate projection, 512 tokens
        {"name": "backward_gate", "kind": "backward", "m": 512, "k": 2048, "n": 8192, "bits": 4, "group": 64},
        # its loss over 512 tokens against a vocabulary of 32000, a tenth of them ignored
        {"name": "loss_512", "kind": "loss", "m": 512, "k": 2048, "n": 32000, "bits": 4, "group": 64},
        # one layer's attention over a 1024-token prompt (32 query heads, 8 kv heads of 64)
        {"name": "attention_prompt", "kind": "attention", "tokens": 1024, "past": 0, "heads": 32, "kv_heads": 8, "head_dim": 64},
        # one layer's attention of a decode step 8191 tokens into a context
        {"name": "attention_step", "kind": "attention", "tokens": 1, "past": 8191, "heads": 32, "kv_heads": 8, "head_dim": 64},
        # a whole request on a 1B decoder: a 512-token prompt, then 32 decode steps
        {"name": "request_1b", "kind": "request", "layers": 16, "dim": 2048, "hidden": 8192, "heads": 32, "kv_heads": 8, "vocab": 32000, "prompt": 512, "steps": 32, "bits": 4, "group": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["linear", "quantize", "backward", "loss", "attention", "request"], [40, 10, 15, 10, 17, 8])[0]
    bits, group = rng.choice([4, 4, 8]), rng.choice([32, 64, 64, 128])
    if kind == "linear":
        m = 1 if rng.random() < 0.25 else _log(rng, 2, 2048)
        k, n = _log(rng, 256, 14336), _log(rng, 64, 40000)
        while m * k * n > 3e10:
            m = max(1, m // 2)
        packed = rng.random() < 0.8
        if packed:  # a model's sizes: whole runs of 32 inputs and of 16 outputs
            k, n = max(128, k // 128 * 128), max(64, n // 16 * 16)
        outs = rng.choice(["%d" % n, "%d" % n, "%d,%d" % (n, n), "%d,%d,%d" % (n, max(64, n // 64 * 16), max(64, n // 64 * 16))])
        if not packed:
            outs = "%d" % n
        return {"kind": kind, "m": m, "k": k, "outs": outs, "bits": bits, "group": group, "packed": packed}
    if kind == "quantize":
        k, n = _log(rng, 256, 14336), _log(rng, 128, 32768)
        return {"kind": kind, "k": k, "n": n if rng.random() < 0.3 else n // 16 * 16, "bits": bits, "group": group}
    if kind == "backward":
        m, k, n = _log(rng, 1, 1024), _log(rng, 256, 8192), _log(rng, 256, 16384)
        while m * k * n > 1.5e10:
            m = max(1, m // 2)
        if rng.random() < 0.7:
            k, n = max(256, k // 64 * 64), max(256, n // 64 * 64)
        return {"kind": kind, "m": m, "k": k, "n": n, "bits": bits, "group": group}
    if kind == "loss":
        m, k, n = _log(rng, 8, 768), _log(rng, 512, 2048), _log(rng, 2048, 32768)
        if rng.random() < 0.7:
            k, n = max(512, k // 64 * 64), max(2048, n // 64 * 64)
        return {"kind": kind, "m": m, "k": k, "n": n, "bits": bits, "group": group}
    if kind == "attention":
        heads, kv_heads, head_dim = rng.choice([(32, 8, 64), (14, 2, 64), (32, 8, 128), (16, 16, 64)])
        tokens = 1 if rng.random() < 0.4 else _log(rng, 2, 1536)
        past = _log(rng, 16, 16384) if tokens == 1 else rng.choice([0, 0, _log(rng, 16, 1024)])
        return {"kind": kind, "tokens": tokens, "past": past, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim}
    dim = rng.choice([512, 896, 1024, 2048])
    heads, kv_heads = {512: (8, 8), 896: (14, 2), 1024: (16, 4), 2048: (32, 8)}[dim]
    return {"kind": kind, "layers": rng.randint(1, 4), "dim": dim, "hidden": rng.choice([2, 4]) * dim, "heads": heads, "kv_heads": kv_heads,
            "vocab": rng.choice([4096, 8000, 32000]), "prompt": _log(rng, 4, 512), "steps": rng.randint(2, 32), "bits": bits, "group": rng.choice([32, 64])}


# ---- device memory shared with torch --------------------------------------------------

class _Shared:
    """What torch needs to see a DeviceBuffer's memory as a tensor (keeps the buffer alive)."""

    def __init__(self, buffer, shape, typestr):
        self.buffer = buffer
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (buffer.ptr, False), "version": 3}


def _view(buffer, shape, typestr="<f4"):
    return torch.as_tensor(_Shared(buffer, shape, typestr), device="cuda")


def _tensor(t):
    """A DeviceTensor holding the fp32 matrix `t`."""
    out = kt.DeviceTensor(kt.DeviceBuffer(t.numel() * 4), t.shape)
    _view(out.buffer, t.shape).copy_(t)
    return out


def _empty(rows, columns):
    return kt.DeviceTensor(kt.DeviceBuffer(rows * columns * 4), (rows, columns))


def _generator(seed, part):
    return torch.Generator(device="cuda").manual_seed((seed * 7919 + part * 104729 + 1) % (1 << 62))


def _normal(seed, part, shape, std=1.0):
    return torch.randn(shape, generator=_generator(seed, part), device="cuda", dtype=torch.float32) * std


def _quantized(w, case, packed=False):
    q = kt.QuantizedTensor.quantize(_tensor(w).buffer, w.shape[0], w.shape[1], kt.Quantization(case["bits"], case["group"]))
    return q.pack() if packed else q


def _outs(case):
    return [int(n) for n in case["outs"].split(",")]


# The inputs of each kind: one function for prepare() and exact().

def _linear_inputs(case, seed):
    k = case["k"]
    ws = [_normal(seed, 10 + i, (k, n), 0.02) for i, n in enumerate(_outs(case))]
    bs = [_normal(seed, 20 + i, (1, n), 0.1) for i, n in enumerate(_outs(case))]
    return _normal(seed, 1, (case["m"], k)), ws, bs


def _backward_inputs(case, seed):
    return _normal(seed, 1, (case["m"], case["n"]), 1e-3), _normal(seed, 2, (case["k"], case["n"]), 0.02)


def _loss_inputs(case, seed):
    hidden, w = _normal(seed, 1, (case["m"], case["k"])), _normal(seed, 2, (case["k"], case["n"]), 0.02)
    rng = np.random.default_rng(seed)
    targets = rng.integers(0, case["n"], case["m"]).astype(np.int32)
    targets[rng.random(case["m"]) < 0.1] = kt.IGNORE_INDEX
    targets[0] = 0  # at least one token counts
    return hidden, w, _normal(seed, 3, (1, case["n"]), 0.1), targets


def _attention_inputs(case, seed):
    t, h, kv, d = case["tokens"], case["heads"], case["kv_heads"], case["head_dim"]
    n = case["past"] + t
    q, k, v = _normal(seed, 1, (t, h * d)), _normal(seed, 2, (1, kv * d)), _normal(seed, 3, (1, kv * d))
    return q, k, v, _normal(seed, 4, (kv, n, d)), _normal(seed, 5, (kv, n, d))


def _request_shapes(case):
    d, h = case["dim"], case["hidden"]
    kv = case["kv_heads"] * (d // case["heads"])
    shapes = {}
    for l in range(case["layers"]):
        for name, shape in (("attention.wQ", (d, d)), ("attention.wK", (d, kv)), ("attention.wV", (d, kv)), ("attention.wOut", (d, d)),
                            ("ffn.wGate", (d, h)), ("ffn.wUp", (d, h)), ("ffn.wDown", (h, d))):
            shapes["block.%d.%s" % (l, name)] = shape
    shapes["lmHead"] = (d, case["vocab"])
    shapes["embedding"] = (case["vocab"], d)
    return shapes


def _request_weight(case, seed, index, shape):
    return _normal(seed, 100 + index, shape, 0.02)


def _request_tokens(case, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(0, case["vocab"], case["prompt"]).tolist(), rng.integers(0, case["vocab"], case["steps"]).astype(np.int32)


# ---- prepare: what the program holds before the call ------------------------------------

def prepare(case, seed):
    state = {"case": case}
    kind = case["kind"]
    if kind == "linear":
        x, ws, bs = _linear_inputs(case, seed)
        state["x"], state["layers"] = _tensor(x), []
        for w, b in zip(ws, bs):
            layer = kt.QuantizedLinear(w.shape[0], w.shape[1], kt.Quantization(case["bits"], case["group"]))
            layer.weight, layer.bias = _quantized(w, case, case["packed"]), _tensor(b)
            state["layers"].append(layer)
        state["y"] = [_empty(case["m"], n) for n in _outs(case)]
    elif kind == "quantize":
        k, n, bits = case["k"], case["n"], case["bits"]
        groups, bpr = -(-k // case["group"]), (n + 1) // 2 if bits == 4 else n
        state["w"] = _tensor(_normal(seed, 1, (k, n), 0.02))
        state["q"], state["s"] = kt.DeviceBuffer(k * bpr), _empty(groups, n)
        state["z"] = kt.DeviceBuffer(groups * n) if bits == 4 else None
        state["shapes"] = (k, bpr), (groups, n)
    elif kind == "backward":
        dy, w = _backward_inputs(case, seed)
        state["dy"], state["w"], state["dx"] = _tensor(dy), _quantized(w, case), _empty(case["m"], case["k"])
    elif kind == "loss":
        hidden, w, bias, targets = _loss_inputs(case, seed)
        head = kt.QuantizedLinear(case["k"], case["n"], kt.Quantization(case["bits"], case["group"]))
        head.weight, head.bias = _quantized(w, case, True), _tensor(bias)
        state.update(hidden=_tensor(hidden), head=head, targets=targets, dh=_empty(case["m"], case["k"]), db=_empty(1, case["n"]))
    elif kind == "attention":
        q, k, v, keys, values = _attention_inputs(case, seed)
        state.update(q=_tensor(q), k=_tensor(k), v=_tensor(v), context=_empty(case["tokens"], case["heads"] * case["head_dim"]))
        cache = kt.KVCache(1, case["kv_heads"], case["past"] + case["tokens"], case["head_dim"])
        _view(cache.keys, keys.shape).copy_(keys)
        _view(cache.values, values.shape).copy_(values)
        cache.advance(case["past"])
        freq = np.empty(case["head_dim"] // 2, np.float32)
        _lib.call("kt_rope_inv_freq", case["head_dim"], ctypes.c_float(10000.0), ctypes.c_float(0.0), ctypes.c_float(1.0), ctypes.c_float(4.0), 8192,
                  freq.ctypes.data_as(ctypes.c_void_p))
        state.update(cache=cache, freq=kt.DeviceBuffer.from_numpy(freq))
    elif kind == "request":
        model = kt.Transformer(case["vocab"], case["dim"], case["layers"], case["heads"], case["hidden"], case["kv_heads"],
                               quantization=kt.Quantization(case["bits"], case["group"]), seed=None)
        for i, (name, shape) in enumerate(_request_shapes(case).items()):
            model.set_weight(name, _quantized(_request_weight(case, seed, i, shape), case))
        length = case["prompt"] + case["steps"] + 1
        prompt, forced = _request_tokens(case, seed)
        stream = kt.Stream.create()
        cache, buffers = model.new_cache(length, stream), model.new_inference_buffers(length)
        torch.cuda.synchronize()
        model.prefill(prompt, cache, buffers, stream)  # sizes the stream's workspaces
        model.decode_step(cache, buffers, stream)
        graph = model.capture_decode(cache, buffers, stream)
        stream.synchronize()
        state.update(model=model, stream=stream, cache=cache, buffers=buffers, graph=graph, prompt=prompt, forced=forced,
                     first=kt.DeviceBuffer(case["vocab"] * 4))
    torch.cuda.synchronize()
    return state


# ---- run: one pass ----------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        if len(state["layers"]) == 1:
            state["layers"][0].forward_into(state["x"], state["y"][0])
        else:
            kt.forward_into_group(state["layers"], state["x"], state["y"])
        return [_view(y.buffer, y.shape) for y in state["y"]]
    if kind == "quantize":
        z = state["z"]
        _lib.call("kt_quantize", state["w"].ptr, case["k"], case["n"], case["bits"], case["group"], state["q"].ptr, state["s"].ptr, z.ptr if z else None, None)
        packed, groups = state["shapes"]
        out = {"q": _view(state["q"], packed, "|u1"), "s": _view(state["s"].buffer, groups)}
        if z:
            out["z"] = _view(z, groups, "|u1")
        return out
    if kind == "backward":
        kt.MatMul.multiply_by_quantized_transposed(state["dy"], state["w"], state["dx"], case["m"], accumulate=False)
        return _view(state["dx"].buffer, state["dx"].shape)
    if kind == "loss":
        r = kt.fused_cross_entropy_loss(state["hidden"], state["head"], state["targets"], hidden_grad=state["dh"], bias_grad=state["db"])
        return {"loss": _view(r.loss_buffer, (1,)), "hidden": _view(r.hidden_grad.buffer, r.hidden_grad.shape), "bias": _view(r.bias_grad.buffer, r.bias_grad.shape)}
    if kind == "attention":
        cache, n = state["cache"], case["past"] + case["tokens"]
        if case["tokens"] == 1:
            _lib.call("kt_rope_attention", state["q"].ptr, state["k"].ptr, state["v"].ptr, state["freq"].ptr, 1, cache.position.ptr, n, cache.keys.ptr,
                      cache.values.ptr, 0, n, case["heads"], case["kv_heads"], case["head_dim"], state["context"].ptr, None)
        else:
            _lib.call("kt_attention", state["q"].ptr, case["tokens"], cache.position.ptr, n, cache.keys.ptr, cache.values.ptr, 0, n, case["heads"],
                      case["kv_heads"], case["head_dim"], state["context"].ptr, None)
        out = [_view(state["context"].buffer, state["context"].shape)]
        if case["tokens"] == 1:  # the cache with this step's key and value
            out += [_view(b, (case["kv_heads"], n, case["head_dim"])) for b in (cache.keys, cache.values)]
        return out
    model, stream, cache, buffers = state["model"], state["stream"], state["cache"], state["buffers"]
    cache.reset(stream)
    model.prefill(state["prompt"], cache, buffers, stream)
    state["first"].copy_from(buffers.logits, stream)
    for i in range(case["steps"]):  # the caller's tokens, as in scoring or constrained decoding
        buffers.tokens.upload(state["forced"][i:i + 1], stream)
        state["graph"].replay(1)
    shape = (cache.num_layers, cache.num_heads, cache.max_sequence_length, cache.head_dim)
    return {"first": _view(state["first"], (case["vocab"],)), "logits": _view(buffers.logits, (case["vocab"],)),
            "keys": _view(cache.keys, shape), "values": _view(cache.values, shape)}


# ---- work: what a pass cannot do without -------------------------------------------------

def _weight_bytes(k, n, bits, group):
    groups = -(-k // group)
    return k * ((n + 1) // 2 if bits == 4 else n) + groups * n * (5 if bits == 4 else 4)


def work(case):
    kind = case["kind"]
    if kind == "attention":
        t, past, h, kv, d = (case[x] for x in ("tokens", "past", "heads", "kv_heads", "head_dim"))
        pairs = t * past + t * (t + 1) // 2  # (token, key) pairs of a head
        return {"bytes": 4.0 * (2 * t * h * d + 2 * kv * (past + t) * d), "flops": 4.0 * pairs * h * d}
    b, g = case["bits"], case["group"]
    if kind == "linear":
        m, k = case["m"], case["k"]
        return {"bytes": 4.0 * m * k + sum(_weight_bytes(k, n, b, g) + 4.0 * m * n + 4.0 * n for n in _outs(case)), "flops": sum(2.0 * m * k * n for n in _outs(case))}
    if kind == "request":
        p, s = case["prompt"], case["steps"]
        weights = {name: shape for name, shape in _request_shapes(case).items() if name != "embedding"}
        layers = sum(k * n for name, (k, n) in weights.items() if name != "lmHead")
        head = case["dim"] * case["vocab"]
        keys = p * (p + 1) // 2 + sum(p + i + 1 for i in range(s))
        flops = 2.0 * layers * (p + s) + 2.0 * head * (1 + s) + 4.0 * keys * case["dim"] * case["layers"]
        kv = 2 * 4.0 * case["layers"] * case["kv_heads"] * (case["dim"] // case["heads"])
        return {"bytes": (1 + s) * float(sum(_weight_bytes(k, n, b, g) for k, n in weights.values())) + kv * sum(p + i + 1 for i in range(s)) + kv * (p + s), "flops": flops}
    k, n = case["k"], case["n"]
    if kind == "quantize":
        return {"bytes": 4.0 * k * n + _weight_bytes(k, n, b, g), "flops": 2.0 * k * n}
    m = case["m"]
    if kind == "backward":
        return {"bytes": 4.0 * m * (k + n) + _weight_bytes(k, n, b, g), "flops": 2.0 * m * k * n}
    return {"bytes": 8.0 * m * k + 8.0 * n + _weight_bytes(k, n, b, g), "flops": 4.0 * m * k * n}  # loss


def tolerance(case):
    """About four times what each path measures against its 64-bit result: fp32 sums for up
    to 16 rows, for the transposed product, for the attention and for widths that are not
    whole groups of 8 (4-bit) or 4 columns; fp16 operands with fp32 sums for the other
    products of more rows, and so for the logits of a loss and of a whole model."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "backward":
        return {"rel": 5e-7}
    if kind == "attention":
        return {"rel": 1.4e-6}
    if kind == "linear":
        if case["m"] == 1:
            return {"rel": 1e-6}
        odd = any(n % (8 if case["bits"] == 4 else 4) for n in _outs(case))
        return {"rel": 5e-6 if case["m"] <= 16 else 2e-6 if odd else 1.5e-3}
    if kind == "loss":
        return {"rel": 2e-5}
    return {"rel": 1e-2}


# ---- exact: the same results in 64 bits, from torch alone -------------------------------

def _round(x):
    """Nearest, ties up (the format's rounding), of fp32 values, in 64 bits."""
    return torch.floor(x.double() + 0.5)


def _divide(a, b):
    """The correctly rounded fp32 quotient (of 64 bits rounded once more, which is the same)."""
    return (a.double() / b).float()


def _scheme(w, bits, group):
    """(raw minus zero point [K x N] fp64, scales [G x N] fp32) of a quantized fp32 weight."""
    k, n = w.shape
    groups = -(-k // group)
    q, scales = torch.empty((k, n), dtype=torch.float64, device=w.device), torch.empty((groups, n), dtype=torch.float32, device=w.device)
    pad = torch.cat([w, w[-1:].expand(groups * group - k, n)]) if groups * group != k else w
    blocks = pad.view(groups, group, n)
    if bits == 8:
        mx = blocks.abs().amax(1)
        scales = torch.where(mx > 0, _divide(mx, 127.0), torch.ones_like(mx))
        zeros = torch.zeros_like(scales).double()
        lo, hi = -127.0, 127.0
    else:
        mn, mx = blocks.amin(1).clamp(max=0.0), blocks.amax(1).clamp(min=0.0)
        scales = torch.where(mx - mn > 0, _divide(mx - mn, 15.0), torch.ones_like(mx))
        zeros = _round(_divide(-mn, scales)).clamp(0, 15)
        lo, hi = 0.0, 15.0
    inverse = _divide(torch.ones_like(scales), scales)
    for i in range(groups):
        rows = slice(i * group, min(k, (i + 1) * group))
        q[rows] = (_round(w[rows] * inverse[i]) + zeros[i]).clamp(lo, hi) - zeros[i]
    return q, scales


def _dequantized(w, case):
    q, scales = _scheme(w, case["bits"], case["group"])
    for i in range(scales.shape[0]):
        q[i * case["group"]:(i + 1) * case["group"]] *= scales[i].double()
    return q


def _attend(q, keys, values, past, heads, kv_heads):
    """Causal attention of q [T x heads * d] over keys and values [kv_heads x n x d], fp64."""
    t, d = q.shape[0], keys.shape[2]
    out = torch.empty_like(q)
    n = past + t
    mask = torch.arange(n, device=q.device)[None, :] > past + torch.arange(t, device=q.device)[:, None]
    for h in range(heads):
        kv = h // (heads // kv_heads)
        scores = q[:, h * d:(h + 1) * d] @ keys[kv, :n].t().contiguous() / math.sqrt(d)
        scores = scores.masked_fill(mask, float("-inf"))
        out[:, h * d:(h + 1) * d] = torch.softmax(scores, 1) @ values[kv, :n]
    return out


def _rope(x, first, d, theta):
    """Rotates the pairs (i, i + d / 2) of each head of x [T x heads * d] by position."""
    t = x.shape[0]
    # the model's angles: an fp32 frequency times the position, rounded to fp32
    freq = 1.0 / (theta ** (torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)).float()
    angle = ((first + torch.arange(t, device=x.device, dtype=torch.float32))[:, None] * freq).double()
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x.view(t, -1, d)[..., :d // 2], x.view(t, -1, d)[..., d // 2:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1).reshape(t, -1)


def _norm(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _exact_request(case, seed):
    prompt, forced = _request_tokens(case, seed)
    tokens = prompt + forced.tolist()
    t, p, heads, kv_heads = len(tokens), case["prompt"], case["heads"], case["kv_heads"]
    d = case["dim"] // heads
    shapes = _request_shapes(case)
    index = {name: i for i, name in enumerate(shapes)}

    def weight(name):
        return _dequantized(_request_weight(case, seed, index[name], shapes[name]), case)

    x = weight("embedding")[tokens]
    keys = torch.zeros((case["layers"], kv_heads, t + 1, d), dtype=torch.float64, device=x.device)
    values = torch.zeros_like(keys)
    for l in range(case["layers"]):
        block = "block.%d." % l
        y = _norm(x)
        q, k, v = (y @ weight(block + "attention." + name) for name in ("wQ", "wK", "wV"))
        q, k = _rope(q, 0, d, 10000.0), _rope(k, 0, d, 10000.0)
        keys[l, :, :t], values[l, :, :t] = k.view(t, kv_heads, d).transpose(0, 1), v.view(t, kv_heads, d).transpose(0, 1)
        x = x + _attend(q, keys[l], values[l], 0, heads, kv_heads) @ weight(block + "attention.wOut")
        y = _norm(x)
        x = x + (torch.nn.functional.silu(y @ weight(block + "ffn.wGate")) * (y @ weight(block + "ffn.wUp"))) @ weight(block + "ffn.wDown")
    head = weight("lmHead")
    # the row past the last position holds what an earlier pass left there
    return {"first": _norm(x[p - 1]) @ head, "logits": _norm(x[t - 1]) @ head, "keys": None, "values": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, ws, bs = _linear_inputs(case, seed)
        return [x.double() @ _dequantized(w, case) + b.double() for w, b in zip(ws, bs)]
    if kind == "quantize":
        w = _normal(seed, 1, (case["k"], case["n"]), 0.02)
        return {"q": None, "s": _scheme(w, case["bits"], case["group"])[1].double(), "z": None}
    if kind == "backward":
        dy, w = _backward_inputs(case, seed)
        return dy.double() @ _dequantized(w, case).t().contiguous()
    if kind == "loss":
        hidden, w, bias, targets = _loss_inputs(case, seed)
        w, active = _dequantized(w, case), np.flatnonzero(targets != kt.IGNORE_INDEX)
        rows, wanted = torch.from_numpy(active).cuda(), torch.from_numpy(targets[active].astype(np.int64)).cuda()
        logp = torch.log_softmax(hidden[rows].double() @ w + bias.double(), 1)
        grad = logp.exp()
        grad[torch.arange(len(active), device="cuda"), wanted] -= 1.0
        grad /= len(active)
        dh = torch.zeros(hidden.shape, dtype=torch.float64, device="cuda")
        dh[rows] = grad @ w.t().contiguous()
        return {"loss": -logp[torch.arange(len(active), device="cuda"), wanted].mean().view(1), "hidden": dh, "bias": grad.sum(0, keepdim=True)}
    if kind == "attention":
        q, k, v, keys, values = (t.double() for t in _attention_inputs(case, seed))
        if case["tokens"] == 1:
            d, at = case["head_dim"], case["past"]
            q, k = _rope(q, at, d, 10000.0), _rope(k, at, d, 10000.0)
            keys[:, at], values[:, at] = k.view(-1, d), v.view(-1, d)
            return [_attend(q, keys, values, at, case["heads"], case["kv_heads"]), keys, values]
        return [_attend(q, keys, values, case["past"], case["heads"], case["kv_heads"])]
    return _exact_request(case, seed)
