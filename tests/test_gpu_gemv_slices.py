"""Quantized MatMulNT of 1 to 4 rows whose activations exceed the fused
GEMV's LDS (m * k > 32768): k in slices, in the kernel's form for up to four
rows, against float64. The limbs keep 22 bits below a 256-element chunk's
maximum and the groups' sums add in f32: (k / 64 + 8) roundings of 2^-22."""
import numpy as np
import pytest

from starlight_amd import quant
from starlight_amd.ir import BufferRef, Op, QuantFormat, Value

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [QuantFormat.INT4, QuantFormat.INT8])
@pytest.mark.parametrize("m,k,n,group", [(3, 14336, 300, 128), (4, 14336, 33, 64), (4, 8448, 520, 128),
                                         (3, 11008, 64, 64), (4, 16384, 17, 256), (4, 28672, 48, 128),
                                         (1, 33024, 300, 128), (1, 57344, 33, 64), (2, 16640, 520, 128),
                                         (2, 28672, 130, 64), (2, 32768, 17, 512)])
def test_up_to_four_rows_in_slices(hip, fmt, m, k, n, group):
    r = np.random.default_rng(m + n + k)
    x = (r.standard_normal((m, k)) * 10.0 ** r.uniform(-4, 3, (m, 1))).astype(np.float32)
    top = 8 if fmt == QuantFormat.INT4 else 128
    codes = r.integers(-top, top, (n, k)).astype(np.int8)
    scales = r.uniform(0.001, 0.02, (n, k // group)).astype(np.float32)
    words = quant.pack_codes(codes, fmt)
    wb, sb = hip.upload_new_u32(words), hip.upload_new_f32(scales.ravel())
    hip.bind_quantized(wb, sb, fmt, group, n, k)
    resid = r.standard_normal(m * n).astype(np.float32)
    X = BufferRef(hip.upload_new_f32(x), 0, m * k)
    R = BufferRef(hip.upload_new_f32(resid), 0, m * n)
    Y, Z = (BufferRef(hip.allocate_f32(m * n, 256), 0, m * n) for _ in range(2))
    yv = Value.f32([m, n])
    before = hip.stats()["fused_commands"]
    hip.dispatch(Op.matmul_nt(), [X, BufferRef(wb, 0, words.size)], [Value.f32([m, k]), Value.quantized([n, k], fmt, group)],
                 [Y], [yv])
    hip.dispatch(Op.add(), [R, Y], [yv, yv], [Z], [yv])
    hip.synchronize()
    # (11008 is 43 x 256: no slice count within the limit, so the commands run on their own)
    assert hip.stats()["fused_commands"] - before == (0 if k == 11008 else 2)
    got = hip.read_f32(Y.buffer, m * n).reshape(m, n)
    deq = codes.astype(np.float64) * np.repeat(scales.astype(np.float64), group, axis=1)
    x64 = x.astype(np.float64)
    peak = np.repeat(np.abs(x64).reshape(m, k // 256, 256).max(axis=2), 256, axis=1)
    bound = (k / 64 + 8) * 2.0**-22 * (np.abs(x64) @ np.abs(deq).T) + 2.0**-22 * (peak @ np.abs(deq).T)
    assert np.all(np.abs(got - x64 @ deq.T) <= bound)
    np.testing.assert_array_equal(hip.read_f32(Z.buffer, m * n), resid + got.ravel())
