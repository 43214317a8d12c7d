"""Prefill attention on the bf16 matrix cores, against float64.

A score is off by at most (D + 16) roundings of 2^-24 of scale * sum |q||k|, a
weight by twice the largest such error relative, an output sum by one rounding
per 8 keys and a few for the softmax; all of sum p|v|.
"""
import math

import numpy as np
import pytest

from starlight_amd.device import HipDevice
from starlight_amd.ir import BufferRef, Op, Value, ValueRole

pytestmark = pytest.mark.gpu


def attend(dev, q, k, v, cache, past, scale=None):
    (B, H, S, D), Hkv, max_seq = q.shape, k.shape[1], cache.shape[3]
    scale = 1.0 / math.sqrt(D) if scale is None else scale
    refs = [BufferRef(dev.upload_new_f32(x.ravel()), 0, x.size) for x in (q, k, v, cache)]
    out = BufferRef(dev.allocate_f32(q.size, 256), 0, q.size)
    dev.dispatch(Op.causal_attention(0, H, Hkv, D, scale), refs,
                 [Value.f32(q.shape), Value.f32(k.shape), Value.f32(v.shape),
                  Value.f32(cache.shape, ValueRole.STATE)], [out], [Value.f32(q.shape)], [past])
    return dev.read_f32(out.buffer, q.size).reshape(q.shape)


def inputs(B, H, Hkv, S, past, D, max_seq):
    r = np.random.default_rng(S * 1009 + past * 31 + D + H)
    q = r.standard_normal((B, H, S, D)).astype(np.float32) * 2
    k, v = (r.standard_normal((B, Hkv, S, D)).astype(np.float32) for _ in range(2))
    return q, k, v, r.standard_normal((B, 1, 2, max_seq, Hkv, D)).astype(np.float32)


# query tiles of 64 and their pairs (an odd count, a last tile of one row), key
# tiles of 32 in stages of 64 (remainders of one key, an odd count of tiles),
# keys of earlier calls, heads of 128 from 256 rows, of 64 from 512, shorter the f32 form
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Hkv,S,past,max_seq", [
    (1, 1, 1, 255, 0, 255), (1, 2, 1, 256, 0, 256), (2, 3, 1, 257, 0, 300), (1, 2, 2, 288, 1, 289),
    (2, 4, 2, 320, 33, 384), (1, 2, 1, 321, 31, 352), (1, 8, 2, 300, 77, 400), (1, 2, 1, 256, 1000, 1256),
    (1, 2, 1, 511, 0, 511), (1, 3, 1, 512, 40, 552), (2, 1, 1, 577, 0, 577)])
def test_prefill_attention(hip, B, H, Hkv, S, past, max_seq, D):
    q, k, v, cache = inputs(B, H, Hkv, S, past, D, max_seq)
    got = attend(hip, q, k, v, cache, past).astype(np.float64)
    for b in range(B):
        for h in range(H):
            kv = h // (H // Hkv)
            keys, vals = (np.concatenate([cache[b, 0, x, :past, kv], new[b, kv]]).astype(np.float64)
                          for x, new in ((0, k), (1, v)))
            q64, scale = q[b, h].astype(np.float64), 1.0 / math.sqrt(D)
            seen = np.arange(past + S)[None] <= past + np.arange(S)[:, None]
            s = np.where(seen, q64 @ keys.T * scale, -np.inf)
            p = np.exp(s - s.max(axis=1, keepdims=True))
            p /= p.sum(axis=1, keepdims=True)
            score = (D + 16) * 2.0**-24 * scale * np.max(np.where(seen, np.abs(q64) @ np.abs(keys).T, 0), axis=1)
            bound = (2 * score + ((past + S) / 8 + 64) * 2.0**-24)[:, None] * (p @ np.abs(vals))
            assert np.all(np.abs(got[b, h] - p @ vals) <= bound), (b, h)


# a value that its parts cannot hold is left to the f32 form: the same bits as
# from a device without room for the parts
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 2.0**56, -3e38, 2.0**-101, 1e-42])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("D", [64, 128])
def test_values_out_of_range(hip, monkeypatch, D, where, value):
    q, k, v, cache = inputs(1, 2, 1, 520, 0, D, 2048)
    {"q": q[0, 1], "k": k[0, 0], "v": v[0, 0]}[where][3, 5] = value
    monkeypatch.setenv("SL_HIP_WORKSPACE_BYTES", "65536")
    small = HipDevice(0)
    try:
        want, got = attend(small, q, k, v, cache, 0), attend(hip, q, k, v, cache, 0)
    finally:
        small.close()
    # (q: the block of query tiles 0 and 8 of its head)
    rows = np.r_[0:64, 512:520] if where == "q" else np.r_[0:520]
    heads = [1] if where == "q" else [0, 1]
    for h in heads:
        assert np.array_equal(got[0, h, rows], want[0, h, rows], equal_nan=True)


# scores far apart and large: each query takes exactly the value of the visible
# key with the largest score (the next is M^2 D / 1024 of scale away, the error of
# a score at most (D + 16) 2^-24 of M^2 D)
@pytest.mark.parametrize("M", [1e3, 1e5, 1e8, 2.0**55])
@pytest.mark.parametrize("past", [0, 70])
@pytest.mark.parametrize("D", [64, 128])
def test_large_scores(hip, D, past, M):
    S, max_seq = 520, 640
    q, k, v, cache = inputs(1, 2, 1, S, past, D, max_seq)
    r = np.random.default_rng(D + past)
    sign = r.choice([-1.0, 1.0], D)
    size = r.permutation(past + S) / 1024 + 1 / 1024
    q[:] = sign * M
    cache[0, 0, 0, :past, 0], k[0, 0] = np.split((size[:, None] * sign * M).astype(np.float32), [past])
    vals = np.concatenate([cache[0, 0, 1, :past, 0], v[0, 0]])
    got = attend(hip, q, k, v, cache, past)
    best = [int(np.argmax(size[:past + t + 1])) for t in range(S)]
    assert np.all(np.abs(got - vals[best]) <= 2.0**-22 * np.abs(vals[best]))


# one element of K at 2^40 decides the queries after it by its sign: that key
# alone, or the others without it
@pytest.mark.parametrize("D", [64, 128])
def test_one_large_key(hip, D):
    S, at = 520, 100
    q, k, v, cache = inputs(1, 1, 1, S, 0, D, S)
    q[0, 0, :, 7] = np.where(np.arange(S) % 2, 1.5, -1.5)
    k[0, 0, at, 7] = 2.0**40
    got = attend(hip, q, k, v, cache, 0)[0, 0].astype(np.float64)
    scale = 1.0 / math.sqrt(D)
    q64, k64, v64 = (x[0, 0].astype(np.float64) for x in (q, k, v))
    seen = np.tril(np.ones((S, S), bool))
    seen[:, at] = False
    s = np.where(seen, q64 @ k64.T * scale, -np.inf)
    p = np.exp(s - s.max(axis=1, keepdims=True))
    p /= p.sum(axis=1, keepdims=True)
    score = (D + 16) * 2.0**-24 * scale * np.max(np.where(seen, np.abs(q64) @ np.abs(k64).T, 0), axis=1)
    bound = (2 * score + (S / 8 + 64) * 2.0**-24)[:, None] * (p @ np.abs(v64))
    alone = (np.arange(S) >= at) & (np.arange(S) % 2 == 1)
    want = np.where(alone[:, None], v64[at], p @ v64)
    bound = np.where(alone[:, None], 2.0**-22 * np.abs(v64[at]), bound)
    assert np.all(np.abs(got - want) <= bound)


# no scale, and one that turns the order of the scores around
@pytest.mark.parametrize("scale", [0.0, -0.0, -0.2])
@pytest.mark.parametrize("D", [64, 128])
def test_scale_sign(hip, D, scale):
    S = 540
    q, k, v, cache = inputs(1, 2, 1, S, 0, D, S)
    got = attend(hip, q, k, v, cache, 0, scale).astype(np.float64)
    k64, v64 = k[0, 0].astype(np.float64), v[0, 0].astype(np.float64)
    seen = np.tril(np.ones((S, S), bool))
    for h in range(2):
        q64 = q[0, h].astype(np.float64)
        s = np.where(seen, q64 @ k64.T * scale, -np.inf)
        p = np.exp(s - s.max(axis=1, keepdims=True))
        p /= p.sum(axis=1, keepdims=True)
        score = (D + 16) * 2.0**-24 * abs(scale) * np.max(np.where(seen, np.abs(q64) @ np.abs(k64).T, 0), axis=1)
        bound = (2 * score + (S / 8 + 64) * 2.0**-24)[:, None] * (p @ np.abs(v64))
        assert np.all(np.abs(got[0, h] - p @ v64) <= bound), h
