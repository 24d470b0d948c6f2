"""forward_into_group's operands, without a device: what it hands to kt_qmatmul_group, and what
it refuses."""
import ctypes
from types import SimpleNamespace

import pytest

from kotensor_amd import _lib, linear
from kotensor_amd.device import DeviceBuffer
from kotensor_amd.matmul import DeviceTensor


def _buffer(address, count):
    buffer = object.__new__(DeviceBuffer)
    buffer.nbytes, buffer._ptr = count * 4, address
    buffer.free = lambda: None  # not the library's memory
    return buffer


def _tensor(address, rows, columns):
    return DeviceTensor(_buffer(address, rows * columns), (rows, columns))


def _layer(k, n, bias):
    return SimpleNamespace(in_size=k, out_size=n, bias=bias, weight=SimpleNamespace(qweight=_lib.QWeight()))


@pytest.fixture
def calls(monkeypatch):
    got = []
    monkeypatch.setattr(_lib, "call", lambda name, *args: got.append((name, args)))
    return got


def test_biases_of_every_kind(calls):
    """A bias is a tensor, a buffer, an address or None, as forward_into takes them."""
    layers = [_layer(8, 4, b) for b in (_tensor(0x100, 1, 4), _buffer(0x200, 4), 0x300, None)]
    outs = [_tensor(0x1000 + 256 * i, 2, 4) for i in range(4)]
    assert linear.forward_into_group(layers, _tensor(0x5000, 2, 8), outs) is outs
    (name, args), = calls
    assert name == "kt_qmatmul_group" and args[0] == 0x5000 and args[1] == 2 and args[3] == 4
    assert list(args[4]) == [0x1000, 0x1100, 0x1200, 0x1300]
    assert list(args[5]) == [0x100, 0x200, 0x300, None] and isinstance(args[5][0], (int, ctypes.c_void_p))


def test_buffers_smaller_than_their_shape(calls):
    """A tensor whose buffer was exchanged for a smaller one is refused, input or output."""
    x, out = _tensor(0x5000, 2, 8), _tensor(0x1000, 2, 4)
    for tensor in (x, out):
        whole, tensor.buffer = tensor.buffer, _buffer(0x9000, 4)
        with pytest.raises(_lib.IllegalArgumentException, match="elements, needs"):
            linear.forward_into_group([_layer(8, 4, None)], x, [out])
        tensor.buffer = whole
    with pytest.raises(_lib.IllegalArgumentException, match="differ in length"):
        linear.forward_into_group([_layer(8, 4, None)], x, [])
    assert not calls
