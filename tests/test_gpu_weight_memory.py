"""Device memory of the quantized weights' private copies: given back when a
weight is bound anew and with the device."""
import ctypes

import numpy as np
import pytest

from starlight_amd import quant
from starlight_amd.device import HipDevice, load_library
from starlight_amd.ir import QuantFormat

pytestmark = pytest.mark.gpu


def memory():
    """(free, total) bytes of the GPU, from the runtime that the library uses."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert load_library().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value, total.value


def free_bytes():
    return memory()[0]


def bind(dev, n, k, fmt, payload=None, scales=None, group=128):
    payload = dev.allocate_u32(quant.payload_words(fmt, n, k), 256) if payload is None else payload
    scales = dev.allocate_f32(n * (k // group), 256) if scales is None else scales
    dev.bind_quantized(payload, scales, fmt, group, n, k)
    return payload, scales


def test_copies_are_given_back():
    HipDevice(0).close()  # what a first device leaves loaded
    before = free_bytes()
    dev = HipDevice(0)
    bind(dev, 1024, 1024, QuantFormat.INT4)  # stays
    # one payload as INT4 [2048 x 4096] and INT8 [1024 x 4096], over and over
    payload, s4 = bind(dev, 2048, 4096, QuantFormat.INT4)
    _, s8 = bind(dev, 1024, 4096, QuantFormat.INT8, payload)
    bind(dev, 2048, 4096, QuantFormat.INT4, payload, s4)
    held = free_bytes()
    for _ in range(40):
        bind(dev, 1024, 4096, QuantFormat.INT8, payload, s8)
        bind(dev, 2048, 4096, QuantFormat.INT4, payload, s4)
    assert free_bytes() >= held
    # more than one slab of each kind
    for _ in range(5):
        bind(dev, 14336, 4096, QuantFormat.INT4)
    dev.close()
    assert free_bytes() >= before - (4 << 20)
