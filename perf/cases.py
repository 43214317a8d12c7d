"""The workloads whose time this repository is judged by.

Every case is llama-dense inference through the engine a program uses
(`NativeEngine.step`, `ContinuousBatcher.step`): a prompt prefilled in one
step, a prompt prefilled in chunks, or decode steps after a prefilled prompt.
The models are the repository's own shapes (TINY, the 1B class, the 8B shape)
with dense f32 weights, the only format every StarLight program accepts, or
group-quantized INT4 / INT8 ones. Two of the listed cases run a whole model;
the others run a few of its layers, so that a call is the layers' work and
not the vocabulary projection's.

A pass returns the logits of every step it makes. Two layers or more make the
last position's logits depend on every position's hidden state and K/V rows,
and a decode or chunked pass makes at least two steps, so that a later one
reads the cache rows an earlier one appended.
"""
from __future__ import annotations

import dataclasses

import numpy as np
import torch

from starlight_amd import device as hipdevice
from starlight_amd import engine, graph
from starlight_amd.device import HipDevice
from starlight_amd.graph import LLAMA_1B_INT4, LLAMA_8B_INT4, TINY
from starlight_amd.ir import QuantFormat, ValueRole
from starlight_amd.paged import ContinuousBatcher, PagedKvCache, PagePool

SHAPES = {"tiny": TINY, "1b": LLAMA_1B_INT4, "8b": LLAMA_8B_INT4}
FORMATS = {"f32": None, "int4": QuantFormat.INT4, "int8": QuantFormat.INT8}
DECODE_STEPS = 2
PAGE = 16


def _case(mode, shape, weights, layers, vocab, batch, seq, past, group=128, dense_head=False, name=None):
    """mode: "prefill" (seq tokens after a cached prefix of `past`, which the
    pass itself runs first as a chunk of its own when it is not 0), "decode"
    (DECODE_STEPS steps after a prompt of `past`) or "paged" (the same, the
    rows at lengths of their own from past / 2 to past)."""
    c = dict(mode=mode, shape=shape, weights=weights, layers=layers, vocab=vocab, batch=batch, seq=seq, past=past,
             group=group, dense_head=dense_head)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest model a program runs: launches and host work count
        _case("decode", "tiny", "f32", 2, 1024, 1, 1, 37, name="decode tiny f32"),
        # a small model decoding on its own, whole
        _case("decode", "1b", "int4", 16, 32000, 1, 1, 512, name="decode 1b int4"),
        # the repository's headline: one user of an 8B model, whole
        _case("decode", "8b", "int4", 32, 128256, 1, 1, 1024, name="decode 8b int4"),
        # unquantized weights, the format every program has
        _case("decode", "1b", "f32", 4, 32000, 1, 1, 300, name="decode 1b f32"),
        # a few users together, 8-bit weights, an f32 lm_head kept unquantized
        _case("decode", "8b", "int8", 2, 8192, 4, 1, 777, dense_head=True, name="decode 8b int8 x4"),
        # continuous batching over pages, rows at lengths of their own
        _case("paged", "8b", "int4", 4, 8192, 8, 1, 1312, name="decode 8b int4 paged x8"),
        # a prompt, unquantized
        _case("prefill", "1b", "f32", 2, 8192, 1, 200, 0, name="prefill 1b f32 200"),
        # the headline's prompt
        _case("prefill", "8b", "int4", 2, 8192, 1, 1024, 0, name="prefill 8b int4 1024"),
        # a short question, of no round length
        _case("prefill", "8b", "int4", 2, 8192, 1, 77, 0, name="prefill 8b int4 77"),
        # 8-bit weights in smaller groups
        _case("prefill", "8b", "int8", 2, 8192, 1, 500, 0, group=64, name="prefill 8b int8 500"),
        # a long document on a small model: attention counts
        _case("prefill", "1b", "int4", 2, 8192, 1, 3001, 0, name="prefill 1b int4 3001"),
        # two prompts together, in chunks: the second chunk attends to the first
        _case("prefill", "8b", "int4", 2, 8192, 2, 256, 640, name="prefill 8b int4 x2 chunked"),
    ]


def _log_between(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    mode = rng.choice(["decode", "decode", "paged", "prefill", "prefill", "prefill"])
    shape = rng.choice(["tiny", "1b", "8b", "8b"])
    weights = "f32" if shape == "tiny" else rng.choice(["f32", "int4", "int4", "int8"])
    if mode == "paged" and shape == "tiny":
        shape, weights = "1b", "int4"
    layers = 2 if shape == "8b" or mode == "prefill" else rng.choice([2, 3, 4])
    vocab = rng.choice([1024, 5000, 8192])
    group = rng.choice([64, 128, 128])
    dense_head = weights != "f32" and rng.random() < 0.25
    if mode == "prefill":
        past = 0
        batch = rng.choice([1, 1, 1, 2, 3])
        most = {"tiny": 2048, "1b": 3000, "8b": 1200}[shape] // batch
        seq = _log_between(rng, 9, most)
        if rng.random() < 0.25:
            past = _log_between(rng, 16, max(16, most - seq))
        return _case(mode, shape, weights, layers, vocab, batch, seq, past, group, dense_head)
    batch = _log_between(rng, 2, 12) if mode == "paged" else rng.choice([1, 1, 2, 3, 5, 8, 16])
    past = _log_between(rng, 20, 1500)
    return _case(mode, shape, weights, layers, vocab, batch, 1, past, group, dense_head)


# ------------------------------------------------------------------ inputs --


def _config(case):
    return dataclasses.replace(SHAPES[case["shape"]], layers=case["layers"], vocab=case["vocab"],
                               quant=FORMATS[case["weights"]], group=case["group"],
                               quant_lm_head=not case["dense_head"])


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 2 + 1)
    return g


def _quantize(w, group, qmax):
    """Codes (int8) and scales of the group-wise convention of
    starlight_amd.quant."""
    n, k = w.shape
    wg = w.view(n, k // group, group)
    scales = wg.abs().amax(dim=2) / qmax
    r = wg / torch.where(scales == 0, torch.ones_like(scales), scales).unsqueeze(2)
    q = torch.clamp(torch.trunc(r + torch.copysign(torch.full_like(r, 0.5), r)), -qmax, qmax)
    return q.view(n, k).to(torch.int8), scales.contiguous()


def _weights(cfg, seed):
    """(spec, tensor) or (spec, (codes, scales)) of every weight in the
    canonical order: projections and embeddings ~N(0, 0.02), norms ~N(1, 0.1)."""
    g = _generator(seed)
    for spec in graph.weight_specs(cfg):
        w = torch.randn(spec.shape, generator=g, device="cuda", dtype=torch.float32)
        if spec.kind == "norm":
            yield spec, w * 0.1 + 1.0
        elif spec.quantized:
            yield spec, _quantize(w * 0.02, cfg.group, 7 if cfg.quant == QuantFormat.INT4 else 127)
        else:
            yield spec, w * 0.02


def _payload(codes, fmt):
    if fmt == QuantFormat.INT8:
        return codes.contiguous().view(torch.int32).view(-1)
    nib = codes.view(torch.uint8) & 0xF
    return (nib[:, 0::2] | (nib[:, 1::2] << 4)).contiguous().view(torch.int32).view(-1)


def _lengths(case):
    """Cached positions of each row when its decode begins."""
    b, p = case["batch"], case["past"]
    if case["mode"] != "paged":
        return [p] * b
    return [p - (p // 2) * (b - 1 - r) // max(b - 1, 1) for r in range(b)]


def _tokens(case, seed):
    """Every row's tokens: the cached positions', then the pass's own."""
    total = case["past"] + (case["seq"] if case["mode"] == "prefill" else DECODE_STEPS)
    return np.random.default_rng([int(seed), 7]).integers(0, case["vocab"], (case["batch"], total)).astype(np.uint32)


def _program(cfg, batch, seq, max_seq, buffers):
    caps = graph.DeviceCapabilities.from_c(hipdevice.capabilities())
    return engine.compile_program(graph.compile_for(graph.lower_llama(cfg, batch, seq, max_seq), caps), buffers)


def _state_value(program):
    return next(i for i, v in enumerate(program.lowered.ir.values) if v.role == ValueRole.STATE)


def prepare(case, seed):
    cfg = _config(case)
    dev = HipDevice(0)
    buffers = {}
    for spec, w in _weights(cfg, seed):
        if spec.quantized:
            codes, scales = w
            buffers[spec.name] = dev.upload_new_u32(_payload(codes, cfg.quant).cpu().numpy().view(np.uint32))
            buffers[spec.scales] = dev.upload_new_f32(scales.cpu().numpy())
        else:
            buffers[spec.name] = dev.upload_new_f32(w.cpu().numpy())
    del w
    tokens = _tokens(case, seed)
    state = dict(case=case, device=dev, tokens=tokens)
    B, S, P, V = case["batch"], case["seq"], case["past"], case["vocab"]
    if case["mode"] == "prefill":
        max_seq = -(-(P + S + DECODE_STEPS) // 64) * 64
        # the prefix chunk and the rest: two programs of one engine
        first = _program(cfg, B, P if P else S, max_seq, buffers)
        second = _program(cfg, B, S, max_seq, buffers) if P else first
        state["engine"] = engine.NativeEngine(dev, first, second, B, max_seq)
        state["out"] = [np.zeros((B, V), np.float32) for _ in range(2 if P else 1)]
        return state
    max_seq = -(-(P + DECODE_STEPS + 1) // 1024) * 1024
    state["out"] = [np.zeros((B, V), np.float32) for _ in range(DECODE_STEPS)]
    if case["mode"] == "decode":
        state["engine"] = engine.NativeEngine(dev, _program(cfg, B, P, max_seq, buffers),
                                              _program(cfg, B, 1, max_seq, buffers), B, max_seq)
        _step(state, 0, 0, P, state["out"][0])
        return state
    pre = engine.NativeEngine(dev, _program(cfg, 1, P, max_seq, buffers), _program(cfg, 1, 1, max_seq, buffers), 1,
                              max_seq)
    dec = engine.NativeEngine(dev, _program(cfg, B, 1, PAGE, buffers), _program(cfg, B, 1, PAGE, buffers), B, PAGE)
    pages = max_seq // PAGE
    pool = PagePool(num_pages=B * pages, page_size=PAGE, pages_per_seq=pages, max_batch=B)
    np.random.default_rng([int(seed), 8]).shuffle(pool.free)
    cache = PagedKvCache(dev, cfg.layers, cfg.kv_heads, cfg.head_dim, pool)
    state["batcher"] = ContinuousBatcher(dev, pre, pre.state_buffer(_state_value(pre.prefill)), max_seq, P, dec,
                                         dec.state_buffer(_state_value(dec.decode_program)), cache, V)
    for r, n in enumerate(_lengths(case)):
        state["batcher"].admit(r, tokens[r, :n])
    return state


def _step(state, mode, start, count, out):
    """One engine step over positions [start, start + count) of every row."""
    B = state["case"]["batch"]
    positions = np.tile(np.arange(start, start + count, dtype=np.uint32), B)
    state["engine"].step(mode, state["tokens"][:, start:start + count], positions, count, start, out.reshape(-1))


def run(state):
    case, out = state["case"], state["out"]
    P, S = case["past"], case["seq"]
    if case["mode"] == "prefill":
        if P:
            _step(state, 0, 0, P, out[0])
            _step(state, 1, P, S, out[1])
        else:
            _step(state, 0, 0, S, out[0])
        return out
    if case["mode"] == "decode":
        for i in range(DECODE_STEPS):
            _step(state, 1, P + i, 1, out[i])
        return out
    batcher, lengths = state["batcher"], _lengths(case)
    for r, n in enumerate(lengths):
        batcher.pool.set_length(r, n)  # every pass decodes the same positions
    for i in range(DECODE_STEPS):
        logits = batcher.step({r: int(state["tokens"][r, n + i]) for r, n in enumerate(lengths)})
        for r in logits:
            out[i][r] = logits[r]
    return out


# ---------------------------------------------------- what a pass is held to --


def _steps(case):
    """(query tokens per row, cached positions of each row) of every step."""
    if case["mode"] == "prefill":
        P, S, B = case["past"], case["seq"], case["batch"]
        return ([(P, [0] * B)] if P else []) + [(S, [P] * B)]
    return [(1, [n + i for n in _lengths(case)]) for i in range(DECODE_STEPS)]


def work(case):
    """Per step: every layer weight and lm_head read once, the cached K/V rows
    read once and the new ones written, the embedding rows, and the logits."""
    cfg = _config(case)
    weight_bytes, layer_values = 0, 0
    for spec in graph.weight_specs(cfg):
        if spec.name == "embed":
            continue
        n = int(np.prod(spec.shape))
        if spec.quantized:
            weight_bytes += n // (2 if cfg.quant == QuantFormat.INT4 else 1) + n // cfg.group * 4
        else:
            weight_bytes += 4 * n
        if spec.kind == "linear" and spec.name != "lm_head":
            layer_values += n
    B, H, V = case["batch"], cfg.hidden, case["vocab"]
    kv_row = cfg.layers * 2 * cfg.kv_heads * cfg.head_dim * 4
    total_bytes, flops = 0, 0
    for count, cached in _steps(case):
        total_bytes += weight_bytes + B * (count * (H * 4 + kv_row) + V * 4) + sum(cached) * kv_row
        pairs = sum(count * n + count * (count + 1) // 2 for n in cached)
        flops += 2 * B * count * layer_values + 2 * B * V * H + 4 * pairs * cfg.heads * cfg.head_dim * cfg.layers
    return {"bytes": total_bytes, "flops": flops}


def tolerance(case):
    """f32 weights, activations and sums throughout: roundings of 2^-24 that a
    few thousand additions and the layers carry on. Measured against `exact`:
    0.7e-6 to 5.4e-6 over the models of 2 to 4 layers, 3.4e-6 over 16 and
    7.0e-6 over 32; four times the largest of each, and five standard
    deviations of that for one logit."""
    rel = 2e-5 if case["layers"] <= 4 else 3e-5
    return {"rel": rel, "max": 5 * rel}


def _attend(q, k, v, first):
    """Causal attention of q [heads, s, d] at positions first .. over k, v
    [kv_heads, first + s, d], in blocks of heads."""
    heads, s, d = q.shape
    per = heads // k.shape[0]
    mask = torch.arange(k.shape[1], device=q.device)[None, :] > first + torch.arange(s, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        scores = (q[h] @ k[h // per].t()) / d**0.5
        scores.masked_fill_(mask, float("-inf"))
        out[h] = torch.softmax(scores, dim=-1) @ v[h // per]
    return out


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps) * w


def exact(case, seed):
    """The same forward pass in float64: every row's whole sequence at once,
    logits at the positions whose steps return them."""
    cfg = _config(case)
    f64 = torch.float64
    tokens = torch.from_numpy(_tokens(case, seed).astype(np.int64)).cuda()
    steps = _steps(case)
    B, D = case["batch"], cfg.head_dim
    rows = [cached_first + sum(c for c, _ in steps) for cached_first in steps[0][1]]  # each row's length
    half = torch.arange(D // 2, device="cuda", dtype=f64)
    angle = torch.arange(max(rows), device="cuda", dtype=f64)[:, None] / float(np.float32(cfg.theta))**(2 * half / D)
    cos, sin = angle.cos(), angle.sin()

    def rope(x):  # [s, heads, d] -> [heads, s, d], NeoX pairs
        x = x.transpose(0, 1)
        c, s = cos[:x.shape[1]], sin[:x.shape[1]]
        lo, hi = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([lo * c - hi * s, lo * s + hi * c], dim=-1)

    h, parts = None, {}
    for spec, w in _weights(cfg, seed):
        if spec.quantized:
            codes, scales = w
            n, k = codes.shape
            w = (codes.view(n, k // cfg.group, cfg.group).to(f64) * scales.to(f64).unsqueeze(2)).view(n, k)
        else:
            w = w.to(f64)
        role = spec.name.rpartition(".")[2] if spec.name.startswith("layers") else spec.name
        if role == "embed":
            h = [w[tokens[b, :rows[b]]] for b in range(B)]
            continue
        parts[role] = w
        eps = float(np.float32(cfg.eps))
        if role == "o":
            for b in range(B):
                x = _norm(h[b], parts["attn_norm"], eps)
                q, k, v = (x @ parts[r].t() for r in ("q", "k", "v"))
                att = _attend(rope(q.view(-1, cfg.heads, D)), rope(k.view(-1, cfg.kv_heads, D)),
                              v.view(-1, cfg.kv_heads, D).transpose(0, 1), 0)
                h[b] = h[b] + att.transpose(0, 1).reshape(rows[b], -1) @ w.t()
            parts = {}
        elif role == "down":
            for b in range(B):
                x = _norm(h[b], parts["mlp_norm"], eps)
                h[b] = h[b] + (torch.nn.functional.silu(x @ parts["gate"].t()) * (x @ parts["up"].t())) @ w.t()
            parts = {}
    out, at = [], list(steps[0][1])
    for count, _ in steps:
        at = [a + count for a in at]
        last = torch.stack([h[b][at[b] - 1] for b in range(B)])
        out.append((_norm(last, parts["final_norm"], float(np.float32(cfg.eps))) @ parts["lm_head"].t()).cpu().numpy())
    return out
