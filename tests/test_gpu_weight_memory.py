"""Device memory of the quantized weights' private copies: given back when a
weight is bound anew and with the device."""
import ctypes

import numpy as np
import pytest

from starlight_amd import quant
from starlight_amd.device import DeviceError, HipDevice, load_library
from starlight_amd.ir import BufferRef, Op, QuantFormat, Value

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


N, K, M = 512, 1024, 48


def products(dev, weight, words, a, times=1):
    out = dev.allocate_f32(M * N, 256)
    ab = dev.upload_new_f32(a)
    for _ in range(times):  # (the third is a captured graph's)
        dev.dispatch(Op.matmul_nt(), [BufferRef(ab, 0, M * K), BufferRef(weight, 0, words)],
                     [Value.f32([M, K]), Value.quantized([N, K], QuantFormat.INT4, 128)],
                     [BufferRef(out, 0, M * N)], [Value.f32([M, N])])
        dev.submit()
    return dev.read_f32(out, M * N)


def inputs():
    r = np.random.default_rng(3)
    words, scales = quant.quantize((r.standard_normal((N, K)) * 0.05).astype(np.float32), 128, QuantFormat.INT4)
    return words, scales, r.standard_normal(M * K).astype(np.float32)


def bound(dev, words, scales):
    return bind(dev, N, K, QuantFormat.INT4, dev.upload_new_u32(words), dev.upload_new_f32(scales))[0]


def test_copies_can_be_declined(monkeypatch):
    """Without the 6-bit copies the same products come from the fp16 route."""
    words, scales, a = inputs()
    results, used = [], []
    for decline in (False, True):
        if decline:
            monkeypatch.setenv("SL_HIP_FP6_COPIES", "0")
        dev = HipDevice(0)
        before = free_bytes()
        results.append(products(dev, bound(dev, words, scales), words.size, a))
        used.append(before - free_bytes())
        dev.close()
    assert used[1] < used[0]
    assert not np.array_equal(results[0], results[1])
    assert np.linalg.norm(results[0] - results[1]) <= 2.0**-21 * np.linalg.norm(results[0])


def test_a_failing_allocation_takes_the_6_bit_copies_back(monkeypatch):
    """An allocation of the whole GPU fails with and without them, but they are
    gone then, nothing else is, and later products are the fp16 route's."""
    words, scales, a = inputs()
    monkeypatch.setenv("SL_HIP_FP6_COPIES", "0")
    dev = HipDevice(0)
    without = products(dev, bound(dev, words, scales), words.size, a)
    dev.close()
    monkeypatch.delenv("SL_HIP_FP6_COPIES")
    dev = HipDevice(0)
    weight = bound(dev, words, scales)
    assert not np.array_equal(products(dev, weight, words.size, a, 3), without)
    free, total = memory()
    with pytest.raises(DeviceError) as e:
        dev.allocate_f32(total // 4, 256)
    assert e.value == DeviceError.out_of_memory(total // 4)
    assert free_bytes() > free
    assert np.array_equal(products(dev, weight, words.size, a, 3), without)
    # bound later: no copy either
    assert np.array_equal(products(dev, bound(dev, words, scales), words.size, a), without)
    dev.close()
