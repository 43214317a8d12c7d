"""Dense f32 MatMulNT: the decode GEMV kernels, the GEMM, and their fusions.

Products against float64 with the bound of f32 summation: a chain of at most
k / 4 + 64 additions rounds each partial sum by 2^-24 of at most sum |a||w|.
"""
import numpy as np
import pytest

import oracle
from conftest import assert_normwise
from starlight_amd.ir import BufferRef, Op, Value, ValueRole

pytestmark = pytest.mark.gpu


def assert_products(got, a, w):
    a64, w64 = a.astype(np.float64), w.astype(np.float64)
    bound = (a.shape[1] / 4 + 64) * 2.0**-24 * (np.abs(a64) @ np.abs(w64).T)
    diff = np.abs(got.astype(np.float64) - a64 @ w64.T)
    assert np.all(diff <= bound + 1e-30), f"largest excess {np.max(diff - bound)}"


def dense(hip, shape, r):
    x = r.uniform(-1, 1, shape).astype(np.float32)
    return x, BufferRef(hip.upload_new_f32(x), 0, x.size)


# m: 1-4 rows in LDS (m * k <= 16384), 5-32 or longer k on the matrix cores,
# 33 the GEMM; k: one float4, less than a wave's batch, its edges, past LDS
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 16, 17, 32, 33])
@pytest.mark.parametrize("k,n", [(4, 1), (12, 33), (252, 15), (256, 16), (1020, 17), (1024, 300), (1028, 100),
                                 (4096, 40), (5464, 9), (16384, 5), (16388, 21)])
def test_few_rows_matmul(hip, m, k, n):
    r = np.random.default_rng(m * 100003 + k * 31 + n)
    a, ar = dense(hip, (m, k), r)
    w, wr = dense(hip, (n, k), r)
    out = hip.allocate_f32(m * n + 8, 256)
    hip.upload_f32(out, np.full(m * n + 8, 7.0, np.float32))
    hip.dispatch(Op.matmul_nt(), [ar, wr], [Value.f32([m, k]), Value.f32([n, k])], [BufferRef(out, 4, m * n)],
                 [Value.f32([m, n])])
    got = hip.read_f32(out, m * n + 8)
    assert np.all(got[:4] == 7.0) and np.all(got[-4:] == 7.0)
    assert_products(got[4:-4].reshape(m, n), a, w)


# row blocks of 16 to 128 rows and their remainders, ragged columns, k tails,
# one slice and several
@pytest.mark.parametrize("m,k,n", [(33, 4, 1), (47, 36, 130), (64, 2048, 128), (100, 2052, 129), (129, 1028, 300),
                                   (200, 8192, 40), (250, 40, 1000), (513, 516, 260), (1030, 128, 2050),
                                   (2100, 64, 4100)])
def test_many_rows_matmul(hip, m, k, n):
    test_few_rows_matmul(hip, m, k, n)


@pytest.mark.parametrize("m,k", [(1, 1000), (6, 1000), (40, 1000)])
def test_infinite_and_nan_weights_stay_in_their_column(hip, m, k):
    """Loads past a row's end are clamped to its last element: an infinity or
    NaN there reaches that row's products only, as the product it is."""
    r = np.random.default_rng(k)
    a, ar = dense(hip, (m, k), r)
    w = r.uniform(-1, 1, (20, k)).astype(np.float32)
    w[3, -1], w[7, -1], w[11, 0] = np.inf, np.nan, -np.inf
    wr = BufferRef(hip.upload_new_f32(w), 0, w.size)
    out = hip.allocate_f32(m * 20, 256)
    hip.dispatch(Op.matmul_nt(), [ar, wr], [Value.f32([m, k]), Value.f32([20, k])], [BufferRef(out, 0, m * 20)],
                 [Value.f32([m, 20])])
    got = hip.read_f32(out, m * 20).reshape(m, 20)
    assert np.array_equal(got[:, 3], np.inf * np.sign(a[:, -1]))
    assert np.all(np.isnan(got[:, 7]))
    assert np.array_equal(got[:, 11], -np.inf * np.sign(a[:, 0]))
    keep = [c for c in range(20) if c not in (3, 7, 11)]
    assert_products(got[:, keep], a, w[keep])


def test_one_weight_for_a_batch_is_more_rows(hip):
    r = np.random.default_rng(5)
    for b, m in ((3, 1), (8, 1), (5, 20)):  # 3, 8 and 100 rows
        a, ar = dense(hip, (b, m, 132), r)
        w, wr = dense(hip, (70, 132), r)
        out = hip.allocate_f32(b * m * 70, 256)
        hip.dispatch(Op.matmul_nt(), [ar, wr], [Value.f32([b, m, 132]), Value.f32([70, 132])],
                     [BufferRef(out, 0, b * m * 70)], [Value.f32([b, m, 70])])
        assert_products(hip.read_f32(out, b * m * 70).reshape(-1, 70), a.reshape(-1, 132), w)


# rows x hidden in LDS with the norm inside the launch (k % 256 == 0), the
# same past LDS or past 4 rows, and k % 256 != 0: the norm as its own launch
@pytest.mark.parametrize("rows,hidden,inter", [(1, 256, 688), (1, 2048, 512), (3, 512, 100), (4, 4096, 64), (4, 8192, 48),
                                               (2, 260, 52), (5, 512, 96), (20, 256, 64),
                                               (40, 256, 64), (130, 2048, 96)])
def test_dense_decode_units_fuse(hip, rows, hidden, inter):
    """RmsNorm + three projections, a projection + Add and, up to 32 rows,
    RmsNorm + SwiGlu + Add run as fused units, every command's output written."""
    r = np.random.default_rng(rows * 7 + hidden)
    x, xr = dense(hip, (rows, hidden), r)
    g, gr = dense(hip, (hidden,), r)
    ns = [hidden, 40, 24]
    ws = [dense(hip, (n, hidden), r) for n in ns]
    gate, up = dense(hip, (inter, hidden), r), dense(hip, (inter, hidden), r)
    down = dense(hip, (hidden, inter), r)
    size = {"normed": hidden, "q": ns[0], "k": ns[1], "v": ns[2], "h2": hidden, "o": hidden, "normed2": hidden,
            "f": hidden, "h3": hidden}
    buf = {name: BufferRef(hip.allocate_f32(rows * n, 256), 0, rows * n) for name, n in size.items()}
    f32 = Value.f32
    act, gv = f32([rows, hidden]), f32([hidden], ValueRole.PARAM)
    before = hip.stats()
    hip.dispatch(Op.rms_norm(1e-5), [xr, gr], [act, gv], [buf["normed"]], [act])
    for name, (w, wr) in zip("qkv", ws):
        hip.dispatch(Op.matmul_nt(), [buf["normed"], wr], [act, f32(w.shape)], [buf[name]], [f32([rows, w.shape[0]])])
    hip.dispatch(Op.matmul_nt(), [buf["q"], ws[0][1]], [act, f32(ws[0][0].shape)], [buf["o"]], [act])
    hip.dispatch(Op.add(), [xr, buf["o"]], [act, act], [buf["h2"]], [act])
    hip.dispatch(Op.rms_norm(1e-5), [buf["h2"], gr], [act, gv], [buf["normed2"]], [act])
    hip.dispatch(Op.swiglu(), [buf["normed2"], gate[1], up[1], down[1]],
                 [act, f32(gate[0].shape), f32(up[0].shape), f32(down[0].shape)], [buf["f"]], [act])
    hip.dispatch(Op.add(), [buf["h2"], buf["f"]], [act, act], [buf["h3"]], [act])
    hip.synchronize()
    assert hip.stats()["fused_commands"] - before["fused_commands"] == (9 if rows <= 32 else 6)
    got = {name: hip.read_f32(b.buffer, b.len) for name, b in buf.items()}
    normed = oracle.rms_norm(x.ravel(), g, rows, hidden, 1e-5)
    assert_normwise(got["normed"], normed)
    for name, (w, _) in zip("qkv", ws):
        assert_normwise(got[name], oracle.matmul_nt(normed, w.ravel(), 1, rows, hidden, w.shape[0]))
    o = oracle.matmul_nt(got["q"], ws[0][0].ravel(), 1, rows, hidden, hidden)
    assert_normwise(got["o"], o)
    assert np.array_equal(got["h2"], x.ravel() + got["o"])
    normed2 = oracle.rms_norm(got["h2"], g, rows, hidden, 1e-5)
    assert_normwise(got["normed2"], normed2)
    f = oracle.swiglu(got["normed2"], gate[0].ravel(), up[0].ravel(), down[0].ravel(), rows, hidden, inter)
    assert_normwise(got["f"], f)
    assert np.array_equal(got["h3"], got["h2"] + got["f"])
    # the same commands on their own kernels
    hip.set_options(fusion=False)
    hip.dispatch(Op.rms_norm(1e-5), [xr, gr], [act, gv], [buf["normed"]], [act])
    hip.dispatch(Op.swiglu(), [buf["normed"], gate[1], up[1], down[1]],
                 [act, f32(gate[0].shape), f32(up[0].shape), f32(down[0].shape)], [buf["f"]], [act])
    hip.synchronize()
    hip.set_options()
    f = oracle.swiglu(normed, gate[0].ravel(), up[0].ravel(), down[0].ravel(), rows, hidden, inter)
    assert_normwise(hip.read_f32(buf["f"].buffer, buf["f"].len), f)


# Every operand of the units off 16-byte alignment in turn (index: floats to
# start at), in the forms with the norm inside the launch, ahead of it, and ahead
# of the GEMM: commands no dense kernel takes as a unit run one by one.
@pytest.mark.parametrize("off", ["x", "gamma", "normed", "w", "gate", "down", "resid", "out"])
@pytest.mark.parametrize("rows,hidden", [(1, 256), (4, 256), (2, 260), (5, 256), (32, 256), (40, 256)])
def test_units_with_an_unaligned_operand(hip, rows, hidden, off):
    r = np.random.default_rng(rows + hidden)
    inter, n = 48, 36

    def put(name, *shape):
        x = r.uniform(-1, 1, shape).astype(np.float32)
        at = 1 if name == off else 0
        return x, BufferRef(hip.upload_new_f32(np.concatenate([np.zeros(at, np.float32), x.ravel()])), at, x.size)

    def room(name, width):
        at = 1 if name == off else 0
        return BufferRef(hip.allocate_f32(rows * width + at, 256), at, rows * width)

    x, xr = put("x", rows, hidden)
    g, gr = put("gamma", hidden)
    (w, wr), (w2, w2r) = put("w", n, hidden), put("", n, hidden)
    (gate, gater), (up, upr), (down, downr) = put("gate", inter, hidden), put("", inter, hidden), put("down", hidden, inter)
    res, resr = put("resid", rows, n)
    res2, res2r = put("resid", rows, hidden)
    normed, one, two, added = room("normed", hidden), room("out", n), room("", n), room("out", n)
    normed2, f, added2 = room("normed", hidden), room("out", hidden), room("out", hidden)
    f32 = Value.f32
    act, gv, on, wv = f32([rows, hidden]), f32([hidden], ValueRole.PARAM), f32([rows, n]), f32([n, hidden])
    hip.dispatch(Op.rms_norm(1e-5), [xr, gr], [act, gv], [normed], [act])
    hip.dispatch(Op.matmul_nt(), [normed, wr], [act, wv], [one], [on])
    hip.dispatch(Op.matmul_nt(), [normed, w2r], [act, wv], [two], [on])
    hip.dispatch(Op.add(), [resr, two], [on, on], [added], [on])
    hip.dispatch(Op.rms_norm(1e-5), [xr, gr], [act, gv], [normed2], [act])
    hip.dispatch(Op.swiglu(), [normed2, gater, upr, downr],
                 [act, f32([inter, hidden]), f32([inter, hidden]), f32([hidden, inter])], [f], [act])
    hip.dispatch(Op.add(), [res2r, f], [act, act], [added2], [act])
    hip.synchronize()

    def got(ref):
        return hip.read_f32(ref.buffer, ref.offset + ref.len)[ref.offset:]

    want = oracle.rms_norm(x.ravel(), g, rows, hidden, 1e-5)
    for ref in (normed, normed2):
        assert_normwise(got(ref), want)
    assert_normwise(got(one), oracle.matmul_nt(want, w.ravel(), 1, rows, hidden, n))
    assert_normwise(got(two), oracle.matmul_nt(want, w2.ravel(), 1, rows, hidden, n))
    assert np.array_equal(got(added), res.ravel() + got(two))
    assert_normwise(got(f), oracle.swiglu(want, gate.ravel(), up.ravel(), down.ravel(), rows, hidden, inter))
    assert np.array_equal(got(added2), res2.ravel() + got(f))


def test_units_with_overlapping_regions_keep_the_command_order(hip):
    """A projection that writes over another's weight, or reads a weight the
    norm before it wrote, gives what the commands give one after the other."""
    r = np.random.default_rng(11)
    k = 256
    x, xr = dense(hip, (1, k), r)
    g, gr = dense(hip, (k,), r)
    w, wr = dense(hip, (8, k), r)
    pool0 = r.uniform(-1, 1, 8 * k).astype(np.float32)
    pool = hip.upload_new_f32(pool0)
    act, gv, wv = Value.f32([1, k]), Value.f32([k], ValueRole.PARAM), Value.f32([8, k])
    out = BufferRef(hip.allocate_f32(8, 256), 0, 8)
    normed = BufferRef(hip.allocate_f32(k, 256), 0, k)
    # the second projection's output lies in the first one's weight
    hip.dispatch(Op.rms_norm(1e-5), [xr, gr], [act, gv], [normed], [act])
    hip.dispatch(Op.matmul_nt(), [normed, BufferRef(pool, 0, 8 * k)], [act, wv], [out], [Value.f32([1, 8])])
    hip.dispatch(Op.matmul_nt(), [normed, wr], [act, wv], [BufferRef(pool, 64, 8)], [Value.f32([1, 8])])
    hip.synchronize()
    n = oracle.rms_norm(x.ravel(), g, 1, k, 1e-5)
    assert_normwise(hip.read_f32(out.buffer, 8), oracle.matmul_nt(n, pool0, 1, 1, k, 8))
    second = oracle.matmul_nt(n, w.ravel(), 1, 1, k, 8)
    after = hip.read_f32(pool, 8 * k)
    assert_normwise(after[64:72], second)
    # the norm's output is row 0 of the weight read next
    hip.dispatch(Op.rms_norm(1e-5), [xr, gr], [act, gv], [BufferRef(pool, 0, k)], [act])
    hip.dispatch(Op.matmul_nt(), [BufferRef(pool, 0, k), BufferRef(pool, k, 4 * k)], [act, Value.f32([4, k])],
                 [BufferRef(out.buffer, 0, 4)], [Value.f32([1, 4])])
    hip.dispatch(Op.matmul_nt(), [xr, BufferRef(pool, 0, 4 * k)], [act, Value.f32([4, k])],
                 [BufferRef(out.buffer, 4, 4)], [Value.f32([1, 4])])
    hip.synchronize()
    after[:k] = n
    got = hip.read_f32(out.buffer, 8)
    assert_normwise(got[:4], oracle.matmul_nt(n, after[k:5 * k], 1, 1, k, 4))
    assert_normwise(got[4:], oracle.matmul_nt(x.ravel(), after[:4 * k], 1, 1, k, 4))
