"""INT4 q-GEMM for many rows on the 6-bit matrix cores, against float64.

Bound: a superblock of 128 k is six or eight products summed in f32 (each
within 2^-22 of the magnitudes it adds) and one multiply-add, superblocks add in
f32, and an activation keeps 29 or 39 bits below the power of two above the
largest of the 32 that share its exponent (half_units).
"""
import numpy as np
import pytest

from starlight_amd import quant
from starlight_amd.device import HipDevice
from starlight_amd.ir import BufferRef, Op, QuantFormat, Value, ValueRole

pytestmark = pytest.mark.gpu


# lane l of a superblock's 128 k holds 16 (i / 4) + 4 l + i % 4, i < 32
LANE_K = np.array([[16 * (i // 4) + 4 * l + i % 4 for i in range(32)] for l in range(4)])


def half_units(a):
    """Largest rounding of each element's digits: half a unit of 2^-29 of its
    block's power of two, of 2^-39 where more than 16 of the 32 are nonzero and
    below 2^-8 of it."""
    m, k = a.shape
    b = np.abs(a.astype(np.float64)).reshape(m, k // 128, 128)[:, :, LANE_K]
    e = np.frexp(b.max(axis=3))[1][..., None]
    further = ((b != 0) & (b < np.ldexp(1.0, e - 8))).sum(axis=3, keepdims=True) > 16
    half = np.ldexp(0.5, e - np.where(further, 39, 29))
    out = np.empty((m, k // 128, 128))
    out[:, :, LANE_K] = half
    return out.reshape(m, k)


def weight(hip, n, k, group, r, codes=None, scales=None):
    """(ref, value, float64 weight) of a bound INT4 weight with codes -8..7."""
    if codes is None:
        codes = r.integers(-8, 8, (n, k)).astype(np.int8)
    if scales is None:
        scales = r.uniform(0.001, 0.05, (n, k // group)).astype(np.float32)
    words = quant.pack_codes(codes, QuantFormat.INT4)
    pb, sb = hip.upload_new_u32(words), hip.upload_new_f32(scales.ravel())
    hip.bind_quantized(pb, sb, QuantFormat.INT4, group, n, k)
    deq = codes.astype(np.float64) * np.repeat(scales.astype(np.float64), group, axis=1)
    return BufferRef(pb, 0, words.size), Value.quantized([n, k], QuantFormat.INT4, group), deq


def run(hip, a, w):
    m, k = a.shape
    wr, wv, deq = w
    n = deq.shape[0]
    out = hip.allocate_f32(m * n, 256)
    hip.upload_f32(out, np.full(m * n, 7.0, np.float32))
    ab = hip.upload_new_f32(a)
    hip.dispatch(Op.matmul_nt(), [BufferRef(ab, 0, m * k), wr], [Value.f32([m, k]), wv], [BufferRef(out, 0, m * n)],
                 [Value.f32([m, n])])
    return hip.read_f32(out, m * n).reshape(m, n)


def assert_products(got, a, deq):
    a64 = a.astype(np.float64)
    m, k = a.shape
    bound = (k / 128 + 8) * 2.0**-22 * (np.abs(a64) @ np.abs(deq).T) + half_units(a) @ np.abs(deq).T
    diff = np.abs(got.astype(np.float64) - a64 @ deq.T)
    assert np.all(diff <= bound + 1e-37), float(np.max(diff - bound))


# m, n around the tiles' edges (32, 64, 128 rows; 128, 256 columns); k of one
# superblock, with and without slices, rows held in 1, 2 and 4 units per
# thread (4096, 8192, 16384) and past them
@pytest.mark.parametrize("m,n,k,group", [
    (17, 1, 128, 128), (31, 15, 256, 128), (33, 127, 384, 128), (64, 129, 1152, 128), (65, 260, 4096, 4096),
    (100, 48, 4224, 128), (129, 16, 8320, 128), (20, 33, 16384, 256), (40, 50, 16512, 128), (300, 520, 512, 256),
    (257, 2050, 640, 128), (520, 4100, 256, 128), (1030, 3000, 384, 128)])
def test_products(hip, m, n, k, group):
    r = np.random.default_rng(m + n + k)
    a = (r.standard_normal((m, k)) * 10.0 ** r.uniform(-6, 3, (m, 1))).astype(np.float32)
    a[3] = 0.0
    w = weight(hip, n, k, group, r)
    got = run(hip, a, w)
    assert np.all(got[3] == 0.0)
    assert_products(got, a, w[2])


def test_elements_far_below_their_row_keep_their_bits(hip):
    """Blocks of a row 2^40 below its maximum are cut at their own exponent:
    with zero codes under the large blocks, the small ones' products remain."""
    r = np.random.default_rng(4)
    m, n, k = 48, 64, 512
    a = r.standard_normal((m, k)).astype(np.float32)
    a[:, :128] *= np.float32(2.0**40)
    codes = r.integers(-8, 8, (n, k)).astype(np.int8)
    codes[:, :128] = 0
    w = weight(hip, n, k, 128, r, codes)
    got = run(hip, a, w)
    assert_products(got, a[:, 128:], w[2][:, 128:])


def outliers(r, m, k, factor, channels):
    a = r.standard_normal((m, k)).astype(np.float32)
    at = {"one": np.arange(77, 78), "each 32": np.arange(7, k, 32),
          "8 of 32": np.flatnonzero(np.arange(k) % 128 % 16 < 4)}[channels]
    a[:, at] *= np.float32(factor)
    return a, at


# Channels far above the others, under zero codes: the others' products keep the
# precision that 22 bits of each element give (2^-22 normwise), as with each
# element split into two fp16 parts. k: rows held by the threads, and longer.
@pytest.mark.parametrize("factor", [30, 1e3, 1e4, 1e5])
@pytest.mark.parametrize("channels", ["one", "each 32", "8 of 32"])
@pytest.mark.parametrize("m,n,k", [(33, 70, 512), (100, 40, 4096), (17, 20, 16512), (130, 300, 256)])
def test_outlier_channels(hip, m, n, k, factor, channels):
    r = np.random.default_rng(k + m)
    a, at = outliers(r, m, k, factor, channels)
    codes = r.integers(-8, 8, (n, k)).astype(np.int8)
    codes[:, at] = 0
    w = weight(hip, n, k, 128, r, codes)
    got = run(hip, a, w)
    want = a.astype(np.float64) @ w[2].T
    assert np.linalg.norm(got - want) <= 2.0**-22 * np.linalg.norm(want)


# Each column one code of 1 under a scale of 1: the activations themselves as the
# digits hold them. Joined from the lowest on, each sum rounds by 2^-24 of itself:
# the last one is the value, the one before at most 16/31 of the highest nonzero
# digit's unit, which is at most 16/15 of the value, the others 1/32 of that.
@pytest.mark.parametrize("kind", ["normal", "silu", "one", "each 32", "8 of 32", "spread", "denormal"])
def test_activations_as_their_digits(hip, kind):
    r = np.random.default_rng(14)
    m, k = 49, 256
    if kind == "normal":
        a = r.standard_normal((m, k))
    elif kind == "silu":
        g = 3 * r.standard_normal((m, k))
        a = g / (1 + np.exp(-g)) * r.standard_normal((m, k))
    elif kind == "spread":
        a = np.ldexp(r.uniform(-1, 1, (m, k)), r.integers(-60, 60, (m, k)))
        a[r.random((m, k)) < 0.2] = 0
    elif kind == "denormal":
        a = np.ldexp(r.uniform(-1, 1, (m, k)), -122 - r.integers(0, 20, (m, k)))
    else:
        a = outliers(r, m, k, 2e3, kind)[0]
    a = a.astype(np.float32)
    w = weight(hip, k, k, 128, r, np.eye(k, dtype=np.int8), np.ones((k, 2), np.float32))
    got = run(hip, a, w).astype(np.float64)
    assert np.all(np.abs(got - a) <= 2.2 * 2.0**-24 * np.abs(a) + half_units(a) + 2.0**-149)


@pytest.mark.parametrize("scale", [1e-42, 1e-37, 1e30, 3e37])
def test_extreme_magnitudes(hip, scale):
    r = np.random.default_rng(9)
    a = (r.uniform(-1, 1, (20, 256)) * scale).astype(np.float32)
    w = weight(hip, 40, 256, 128, r)
    got = run(hip, a, w)
    want = a.astype(np.float64) @ w[2].T
    finite = np.abs(want) < 3.4e38
    err = np.abs(got.astype(np.float64) - want)[finite]
    assert np.all(err <= 1e-5 * np.sqrt(256) * 8 * 0.05 * scale + 2e-45)


# (2^-129 and 2^-128: the smallest and largest maximum with exponent -128)
@pytest.mark.parametrize("top", [2.0**-149, 2.0**-141, 2.0**-129, 1.5 * 2.0**-129, 2.0**-128, 2.0**-126])
def test_zero_blocks_in_a_row_of_denormals(hip, top):
    r = np.random.default_rng(10)
    a = (r.uniform(-1, 1, (20, 384)) * top).astype(np.float32)
    a[:, 5] = top
    a[:, 32:64] = 0.0
    a[:, 128:256] = 0.0
    w = weight(hip, 40, 384, 128, r)
    got = run(hip, a, w)
    want = a.astype(np.float64) @ w[2].T
    # (sums of 224 products of at most 0.4 top, and a result's own rounding)
    assert np.all(np.abs(got - want) <= 224 * 0.4 * top * 2.0**-22 + 2.0**-149)


# a block below 2^-127 of its row's maximum (the first one's, under zero codes)
# may be dropped, but not raised to that
@pytest.mark.parametrize("top,rest", [(1e30, 1e-30), (3e38, 2.0**-3), (1.0, 2.0**-140), (2.0**120, 2.0**-8)])
def test_blocks_below_the_range_of_a_block_scale(hip, top, rest):
    r = np.random.default_rng(12)
    a = (r.uniform(0.5, 1, (20, 256)) * rest).astype(np.float32)
    a[:, :32] = top
    codes = r.integers(1, 8, (24, 256)).astype(np.int8)
    codes[:, :32] = 0
    w = weight(hip, 24, 256, 128, r, codes)
    got = run(hip, a, w)
    want = a.astype(np.float64) @ w[2].T
    assert np.all(got >= 0) and np.all(got <= want * (1 + 2.0**-20) + 2.0**-148)


def test_infinities_and_nan_stay_in_their_row(hip):
    r = np.random.default_rng(6)
    a = r.standard_normal((40, 384)).astype(np.float32)
    a[5, 100], a[17, 383], a[30, 0] = np.inf, np.nan, -np.inf
    w = weight(hip, 70, 384, 128, r)
    got = run(hip, a, w)
    bad = [5, 17, 30]
    assert np.all(np.isnan(got[bad]))
    keep = [i for i in range(40) if i not in bad]
    assert_products(got[keep], a[keep], w[2])


# The rows of a tile past the last one, whose records are not written, hold what an
# earlier call left there: with and without further digits
@pytest.mark.parametrize("m,n,k", [(17, 300, 512), (33, 140, 128), (65, 520, 1024)])
def test_results_do_not_depend_on_earlier_calls(hip, m, n, k):
    r = np.random.default_rng(m)
    a = r.standard_normal((m, k)).astype(np.float32)
    w = weight(hip, n, k, 128, r)
    smooth = r.standard_normal((4 * m, k)).astype(np.float32)
    run(hip, smooth, w)
    first = run(hip, a, w)
    run(hip, outliers(r, 4 * m, k, 1e4, "each 32")[0], w)
    assert np.array_equal(first, run(hip, a, w))


# A device that made no 6-bit copies: the fp16 route, which keeps 22 bits of an
# element down to 2^-40 of its row's largest, whose superblock is 8 products summed
# in f32, and which sums in slices for one weight and for several
@pytest.mark.parametrize("m,n,k,group", [(17, 33, 128, 128), (64, 129, 1152, 128), (65, 260, 4096, 4096),
                                         (77, 128, 14336, 128), (129, 16, 8320, 128), (300, 520, 512, 256),
                                         (520, 4100, 256, 128)])
def test_products_without_the_copies(monkeypatch, m, n, k, group):
    monkeypatch.setenv("SL_HIP_FP6_COPIES", "0")
    dev = HipDevice(0)
    try:
        r = np.random.default_rng(m + n + k)
        a = (r.standard_normal((m, k)) * 10.0 ** r.uniform(-6, 3, (m, 1))).astype(np.float32)
        a[3] = 0.0
        w = weight(dev, n, k, group, r)
        got = run(dev, a, w)
        a64 = np.abs(a.astype(np.float64))
        bound = ((k / 128 + 8) * 2.0**-21 * a64 + 2.0**-40 * a64.max(axis=1, keepdims=True)) @ np.abs(w[2]).T
        assert np.all(np.abs(got.astype(np.float64) - a.astype(np.float64) @ w[2].T) <= bound)
        test_norm_and_three_projections_in_slices(dev, 77, 4096, (300, 129, 65))
    finally:
        dev.close()


def test_reuploaded_payload_and_scales_refresh_the_copy(hip):
    r = np.random.default_rng(8)
    n, k = 48, 256
    a = r.standard_normal((24, k)).astype(np.float32)
    w = weight(hip, n, k, 128, r)
    run(hip, a, w)
    codes = r.integers(-8, 8, (n, k)).astype(np.int8)
    hip.upload_u32(w[0].buffer, quant.pack_codes(codes, QuantFormat.INT4))
    scales = r.uniform(0.001, 0.05, (n, 2)).astype(np.float32)
    hip.upload_f32(w[0].buffer + 1, scales.ravel())
    deq = codes.astype(np.float64) * np.repeat(scales.astype(np.float64), 128, axis=1)
    assert_products(run(hip, a, (w[0], w[1], deq)), a, deq)


@pytest.mark.parametrize("rows,k,ns", [(20, 2048, (64, 32, 32)), (77, 4096, (300, 129, 65)), (140, 512, (256, 16, 48))])
def test_norm_and_three_projections_in_slices(hip, rows, k, ns):
    """One launch for three weights, its k slices' sums added per weight."""
    r = np.random.default_rng(rows)
    x = r.standard_normal((rows, k)).astype(np.float32)
    g = r.uniform(0.5, 1.5, k).astype(np.float32)
    xb, gb = hip.upload_new_f32(x), hip.upload_new_f32(g)
    ws = [weight(hip, n, k, 128, r) for n in ns]
    normed = BufferRef(hip.allocate_f32(rows * k, 256), 0, rows * k)
    outs = [BufferRef(hip.allocate_f32(rows * n, 256), 0, rows * n) for n in ns]
    act = Value.f32([rows, k])
    before = hip.stats()["fused_commands"]
    hip.dispatch(Op.rms_norm(1e-5), [BufferRef(xb, 0, rows * k), BufferRef(gb, 0, k)],
                 [act, Value.f32([k], ValueRole.PARAM)], [normed], [act])
    for (wr, wv, _), out, n in zip(ws, outs, ns):
        hip.dispatch(Op.matmul_nt(), [normed, wr], [act, wv], [out], [Value.f32([rows, n])])
    hip.synchronize()
    assert hip.stats()["fused_commands"] - before == 4
    a = hip.read_f32(normed.buffer, rows * k).reshape(rows, k)
    for (_, _, deq), out, n in zip(ws, outs, ns):
        assert_products(hip.read_f32(out.buffer, rows * n).reshape(rows, n), a, deq)
