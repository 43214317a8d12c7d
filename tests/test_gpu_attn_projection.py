"""The attention unit (SplitHeads x3, Rope x2, CausalAttention, MergeHeads) with
the output projection and its residual Add after it, dense or INT4, against the
oracle run op by op: chained to the decode form for at most 16 rows, run on its
own after the prefill form (16 and more rows of a grouped-query model)."""
import math

import numpy as np
import pytest

import oracle
from conftest import assert_normwise
from starlight_amd import quant
from starlight_amd.ir import BufferRef, Op, QuantFormat, RopeVariant, Value, ValueRole

pytestmark = pytest.mark.gpu

THETA = 500000.0


# off: floats past 16-byte alignment at which the dense weight starts (no dense
# kernel of the unit takes it then). Prompts of 15, 16 and 17 rows lie around
# both the decode form's most and the prefill form's least.
@pytest.mark.parametrize("weight,off", [("dense", 0), ("dense", 1), ("int4", 0)])
@pytest.mark.parametrize("B,H,Hkv,S,past,D,max_seq", [
    (1, 8, 2, 1, 37, 64, 64), (3, 4, 2, 2, 5, 128, 32), (1, 8, 8, 15, 3, 64, 32), (1, 8, 8, 16, 0, 64, 32),
    (1, 8, 2, 16, 0, 64, 32), (1, 4, 2, 16, 9, 128, 64), (1, 4, 1, 17, 0, 64, 32)])
def test_projection_and_add_after_attention(hip, B, H, Hkv, S, past, D, max_seq, weight, off):
    r = np.random.default_rng(H * 100 + S * 10 + D + past)
    n_out, rows = 128, B * S
    sizes = dict(q=rows * H * D, k=rows * Hkv * D, v=rows * Hkv * D, qh=rows * H * D, kh=rows * Hkv * D,
                 vh=rows * Hkv * D, qr=rows * H * D, kr=rows * Hkv * D, att=rows * H * D, merged=rows * H * D,
                 o=rows * n_out, h2=rows * n_out)
    offs, cur = {}, 0
    for name, n in sizes.items():
        offs[name] = cur
        cur += (n + 63) // 64 * 64
    init = np.zeros(cur, np.float32)
    x = {name: r.uniform(-1, 1, sizes[name]).astype(np.float32) for name in "qkv"}
    for name, a in x.items():
        init[offs[name]:offs[name] + a.size] = a
    scratch = hip.upload_new_f32(init)
    ref = {name: BufferRef(scratch, offs[name], n) for name, n in sizes.items()}
    cache = r.uniform(-1, 1, B * 2 * max_seq * Hkv * D).astype(np.float32)
    resid = r.standard_normal(rows * n_out).astype(np.float32)
    pos = np.tile(past + np.arange(S, dtype=np.uint32), B)
    cb, pb, rb = hip.upload_new_f32(cache), hip.upload_new_u32(pos), hip.upload_new_f32(resid)
    lo, hi = offs["qh"], offs["kr"] + sizes["kr"]
    ones = hip.upload_new_f32(np.ones(hi - lo, np.float32))
    w = (r.standard_normal((n_out, H * D)) * 0.05).astype(np.float32)
    if weight == "int4":
        words, scales = quant.quantize(w, 128, QuantFormat.INT4)
        wb = hip.upload_new_u32(words)
        hip.bind_quantized(wb, hip.upload_new_f32(scales), QuantFormat.INT4, 128, n_out, H * D)
        wr, wv = BufferRef(wb, 0, words.size), Value.quantized([n_out, H * D], QuantFormat.INT4, 128)
        w = quant.dequantize(words, scales, n_out, H * D, 128, QuantFormat.INT4)
    else:
        wr = BufferRef(hip.upload_new_f32(np.concatenate([np.zeros(off, np.float32), w.ravel()])), off, w.size)
        wv = Value.f32([n_out, H * D])
    posr = BufferRef(pb, 0, rows)
    qf, kf, hv = Value.f32([B, S, H * D]), Value.f32([B, S, Hkv * D]), Value.f32([B, S, n_out])
    q4, k4, pv = Value.f32([B, H, S, D]), Value.f32([B, Hkv, S, D]), Value.u32([B, S])
    scale = float(np.float32(1.0 / math.sqrt(D)))
    before = hip.stats()["fused_commands"]
    hip.dispatch(Op.split_heads(H, D), [ref["q"]], [qf], [ref["qh"]], [q4])
    hip.dispatch(Op.split_heads(Hkv, D), [ref["k"]], [kf], [ref["kh"]], [k4])
    hip.dispatch(Op.split_heads(Hkv, D), [ref["v"]], [kf], [ref["vh"]], [k4])
    hip.dispatch(Op.rope(RopeVariant.NEOX, THETA), [ref["qh"], posr], [q4, pv], [ref["qr"]], [q4])
    hip.dispatch(Op.rope(RopeVariant.NEOX, THETA), [ref["kh"], posr], [k4, pv], [ref["kr"]], [k4])
    hip.dispatch(Op.causal_attention(0, H, Hkv, D, scale),
                 [ref["qr"], ref["kr"], ref["vh"], BufferRef(cb, 0, cache.size)],
                 [q4, k4, k4, Value.f32([B, 1, 2, max_seq, Hkv, D], ValueRole.STATE)], [ref["att"]], [q4], [past])
    hip.dispatch(Op.merge_heads(H, D), [ref["att"]], [q4], [ref["merged"]], [qf])
    hip.dispatch(Op.matmul_nt(), [ref["merged"], wr], [qf, wv], [ref["o"]], [hv])
    hip.dispatch(Op.add(), [BufferRef(rb, 0, rows * n_out), ref["o"]], [hv, hv], [ref["h2"]], [hv])
    # the split and rotated heads are dead: the unit may leave them unwritten
    hip.dispatch(Op.scale_by(3.0), [BufferRef(ones, 0, hi - lo)], [Value.f32([hi - lo])],
                 [BufferRef(scratch, lo, hi - lo)], [Value.f32([hi - lo])])
    hip.synchronize()
    fused = hip.stats()["fused_commands"] - before
    got = hip.read_f32(scratch, cur)

    qh, kh, vh = (oracle.split_heads(x[name], B, S, heads, D) for name, heads in (("q", H), ("k", Hkv), ("v", Hkv)))
    qr = oracle.rope(qh, pos, B, H, S, D, THETA, "neox")
    kr = oracle.rope(kh, pos, B, Hkv, S, D, THETA, "neox")
    att, want_cache = oracle.causal_attention(qr, kr, vh, cache, B, 1, 0, H, Hkv, S, past, D, max_seq, scale)
    merged = oracle.merge_heads(att, B, S, H, D)
    for name, want in (("att", att), ("merged", merged),
                       ("o", oracle.matmul_nt(merged, w.ravel(), 1, rows, H * D, n_out))):
        assert_normwise(got[offs[name]:offs[name] + sizes[name]], want)
    o = got[offs["o"]:offs["o"] + sizes["o"]]
    np.testing.assert_array_equal(got[offs["h2"]:offs["h2"] + sizes["h2"]], resid + o)
    assert_normwise(hip.read_f32(cb, cache.size), want_cache)
    assert fused == (7 if off else 9)
