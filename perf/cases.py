"""The work a program using dtts has it do, as measurable cases.

A case is a dict of plain values; ``kind`` says which entry point it goes through:

  codec    the codec's waveform stack (``dtts.codec.Codec.decode``), f16 or f32
  unit     one residual unit of that stack (``dtts.nlc.residual_unit``)
  conv     one dilated k=7 conv with its SnakeBeta (``dtts.nlc.conv1d``), as a wide unit's first half
  front    the codec's front half from codes (``dtts.codec_front.CodecFront.decode``)
  step     one decode step of a decoder stack (``dtts.stack.Stack.decode``), replayed as a graph
  prefill  the prompt pass of the same stack (``dtts.stack.Stack.prefill``)

Decoder stacks run a few of their layers: every layer is the same work. Weights are random-init
of the repository's own geometries, drawn with torch's generator from the seed alone, so that
``exact`` can draw the same ones and evaluate the path in float64 with plain torch.
"""
from __future__ import annotations

import math
import os
import sys
from dataclasses import replace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "dream-tts_amd"))

from dtts import codec, codec_front, nlc, ops, stack  # noqa: E402

DEV = "cuda:0"
F16, F32, F64 = torch.float16, torch.float32, torch.float64
GEOMETRY = {"talker": stack.TALKER, "predictor": stack.PREDICTOR}


def listed():
    return [
        # the benchmark's batch: 48 lanes of 5 s of audio at once, f16 storage
        dict(name="codec_f16_48x250", kind="codec", dtype="f16", lanes=48, frames=250),
        # one lane streaming half a second at a time: latency, weights read for few positions
        dict(name="codec_f16_1x25", kind="codec", dtype="f16", lanes=1, frames=25),
        # the reference's own precision for its waveform stack, a small batch
        dict(name="codec_f32_4x250", kind="codec", dtype="f32", lanes=4, frames=250),
        # a residual unit at the third block's width and length, ending in the next SnakeBeta
        dict(name="unit192_16x40000", kind="unit", channels=192, lanes=16, length=40000, dilation=3, snake_out=True),
        # a residual unit at the last block's width, ragged length, plain output
        dict(name="unit96_7x33333", kind="unit", channels=96, lanes=7, length=33333, dilation=9, snake_out=False),
        # the k=7 conv of a second-block unit
        dict(name="conv384_12x10000", kind="conv", channels=384, lanes=12, length=10000, dilation=3),
        # a long document's windows through the front half (300 frames + 25 of context each)
        dict(name="front_10x325", kind="front", lanes=10, frames=325),
        # a talker decode step over a full batch, each lane at its own position
        dict(name="talker_step_48", kind="step", stack="talker", weight="f16", layers=3, lanes=48, cap=1536),
        # the code predictor's step for a single request: the smallest call
        dict(name="predictor_step_1", kind="step", stack="predictor", weight="f16", layers=5, lanes=1, cap=17),
        # a quantized talker at a small batch
        dict(name="talker_step_q8_8", kind="step", stack="talker", weight="q8_0_a32", layers=3, lanes=8, cap=1536),
        # prompts of a batch of requests
        dict(name="talker_prefill_8x256", kind="prefill", layers=2, lanes=8, t=256, start=0),
        # a long prompt (text and reference speech) after a shared prefix, one request
        dict(name="talker_prefill_1x701", kind="prefill", layers=2, lanes=1, t=701, start=37),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["codec", "codec", "unit", "conv", "front", "step", "step", "prefill"])
    if kind == "codec":
        dtype = rng.choice(["f16", "f16", "f32"])
        lanes = _log_int(rng, 1, 48)
        most = (12000 if dtype == "f16" else 4000) // lanes
        return dict(kind=kind, dtype=dtype, lanes=lanes, frames=_log_int(rng, 6, min(400, most)))
    if kind == "unit":
        lanes = _log_int(rng, 1, 48)
        return dict(kind=kind, channels=rng.choice([96, 192]), lanes=lanes,
                    length=_log_int(rng, 100, min(120000, 1000000 // lanes)), dilation=rng.choice([1, 3, 9]),
                    snake_out=rng.random() < 0.5)
    if kind == "conv":
        lanes = _log_int(rng, 1, 48)
        channels = rng.choice([384, 768])
        return dict(kind=kind, channels=channels, lanes=lanes,
                    length=_log_int(rng, 50, min(12000, 300000 // lanes) // (channels // 384)),
                    dilation=rng.choice([1, 3, 9]))
    if kind == "front":
        lanes = _log_int(rng, 1, 48)
        return dict(kind=kind, lanes=lanes, frames=_log_int(rng, 6, min(325, 6000 // lanes)))
    if kind == "step":
        name = rng.choice(["talker", "talker", "predictor"])
        weight = rng.choice(["f16", "f16", "f32", "q8_0", "q8_0_a32"])
        if name == "talker":
            return dict(kind=kind, stack=name, weight=weight, layers=rng.randint(1, 3), lanes=_log_int(rng, 1, 48),
                        cap=_log_int(rng, 128, 1536))
        return dict(kind=kind, stack=name, weight=weight, layers=5, lanes=_log_int(rng, 1, 48), cap=17)
    lanes = _log_int(rng, 1, 16)
    t = _log_int(rng, 8, min(1000, 3000 // lanes))
    return dict(kind=kind, layers=rng.randint(1, 2), lanes=lanes, t=t, start=rng.choice([0, 0, rng.randint(1, 400)]))


# ---------------------------------------------------------------- inputs from the seed alone

class _Draw:
    """torch's generator on the device, one stream per seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEV) * std

    def uniform(self, n, lo, hi):
        return torch.rand(n, generator=self.g, device=DEV) * (hi - lo) + lo

    def ints(self, shape, lo, hi):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV)

    def snake(self, c):
        alpha = self.uniform((c,), 0.5, 1.5)
        return alpha, 1.0 / alpha


def _codec_inputs(case, seed):
    """The stack's weights in checkpoint layouts (unit-gain init, the residual branches damped as
    a trained stack's are) and a latent [lanes, frames, dim]."""
    d, g = _Draw(seed), codec.CONFIG5

    def conv(cout, cin, k, gain=1.0):
        return d.normal((cout, cin, k), gain / math.sqrt(cin * k)), d.normal((cout,), 0.01)

    w = dict(head=conv(g.channels[0], g.latent_dim, g.head_kernel), blocks=[])
    for i, r in enumerate(g.rates):
        cin, cout = g.channels[i], g.channels[i + 1]
        up = d.normal((cin, cout, 2 * r), 1.0 / math.sqrt(cin * 2)), d.normal((cout,), 0.01)
        units = [dict(act1=d.snake(cout), c1=conv(cout, cout, g.ru_kernel, 0.7), act2=d.snake(cout),
                      c2=conv(cout, cout, 1, 0.5)) for _ in g.ru_dilations]
        w["blocks"].append(dict(act=d.snake(cin), up=up, units=units))
    w["out_act"] = d.snake(g.channels[-1])
    w["out"] = conv(1, g.channels[-1], g.out_kernel, 0.5)
    latent = d.normal((case["lanes"], case["frames"], g.latent_dim))
    return w, latent


def _unit_inputs(case, seed):
    d, c = _Draw(seed), case["channels"]
    x = d.normal((case["lanes"], case["length"], c)).half()
    return dict(x=x, act1=d.snake(c), w1=d.normal((c, 7 * c), 1 / math.sqrt(7 * c)).half(), b1=d.normal((c,), 0.01).half(),
                act2=d.snake(c), w2=d.normal((c, c), 1 / math.sqrt(c)).half(), b2=d.normal((c,), 0.01).half(),
                out=d.snake(c))


def _conv_inputs(case, seed):
    d, c = _Draw(seed), case["channels"]
    return dict(x=d.normal((case["lanes"], case["length"], c)).half(),
                w=d.normal((c, 7 * c), 1 / math.sqrt(7 * c)).half(), b=d.normal((c,), 0.01).half(), act=d.snake(c))


def _front_inputs(case, seed):
    d, g = _Draw(seed), codec_front.CODEC
    hw = codec_front.HostWeights()

    def w(shape, fan_in):
        return d.normal(shape, 1 / math.sqrt(fan_in))

    def b(n):
        return d.normal((n,), 0.01)

    hw.codebooks = d.normal((g.n_books, g.book_size, g.book_dim))
    hw.out_proj_sem = w((g.codebook_dim, g.book_dim, 1), g.book_dim)
    hw.out_proj_ac = w((g.codebook_dim, g.book_dim, 1), g.book_dim * 4)
    hw.pre_w, hw.pre_b = w((g.latent_dim, g.codebook_dim, g.pre_kernel), g.codebook_dim * g.pre_kernel), b(g.latent_dim)
    hw.in_w, hw.in_b = w((g.tf_dim, g.latent_dim), g.latent_dim), b(g.tf_dim)
    qw, kvw = g.tf_heads * g.tf_head_dim, g.tf_n_kv * g.tf_head_dim
    for _ in range(g.tf_layers):
        hw.layers.append(dict(
            wq=w((qw, g.tf_dim), g.tf_dim), wk=w((kvw, g.tf_dim), g.tf_dim), wv=w((kvw, g.tf_dim), g.tf_dim),
            wo=w((g.tf_dim, qw), qw), gate=w((g.tf_ffn, g.tf_dim), g.tf_dim), up=w((g.tf_ffn, g.tf_dim), g.tf_dim),
            down=w((g.tf_dim, g.tf_ffn), g.tf_ffn), attn_norm=d.uniform((g.tf_dim,), 0.9, 1.1),
            ffn_norm=d.uniform((g.tf_dim,), 0.9, 1.1), attn_scale=d.uniform((g.tf_dim,), 0.05, 0.15),
            mlp_scale=d.uniform((g.tf_dim,), 0.05, 0.15)))
    hw.tf_norm = d.uniform((g.tf_dim,), 0.9, 1.1)
    hw.out_w, hw.out_b = w((g.latent_dim, g.tf_dim), g.tf_dim), b(g.latent_dim)
    c = g.latent_dim
    for r in g.up_ratios:
        hw.up.append(dict(up_w=w((c, c, r), c), up_b=b(c), dw_w=w((c, 1, g.dw_kernel), g.dw_kernel), dw_b=b(c),
                          ln_w=d.uniform((c,), 0.9, 1.1), ln_b=b(c), pw1_w=w((4 * c, c), c), pw1_b=b(4 * c),
                          pw2_w=w((c, 4 * c), 4 * c), pw2_b=b(c), gamma=d.uniform((c,), 0.05, 0.15)))
    codes = d.ints((case["lanes"], case["frames"], g.n_books), 0, g.book_size)
    return hw, codes


def _q8_0(w):
    """Q8_0 of an [n, k] weight: per 32 values one f16 scale amax / 127 and int8 codes rounded half
    away from zero. Returns (GGML blocks uint8 [n, k/32, 34], the dequantized weight in float64)."""
    n, k = w.shape
    v = w.view(n, k // 32, 32)
    scale = v.abs().amax(-1) / 127
    t = v * torch.where(scale > 0, 1 / scale, scale)[..., None]
    q = (torch.sign(t) * torch.floor(t.abs() + 0.5)).to(torch.int8)
    scale = scale.half()
    blocks = torch.empty((n, k // 32, 34), dtype=torch.uint8, device=w.device)
    blocks[..., :2] = scale.view(torch.uint8).view(n, k // 32, 2)
    blocks[..., 2:] = q.view(torch.uint8)
    return blocks, (q.to(F64) * scale.to(F64)[..., None]).view(n, k)


def _stack_geometry(case):
    g = GEOMETRY[case.get("stack", "talker")]
    return replace(g, layers=case["layers"])


def _stack_weights(d, g):
    """Per layer f32 projections in the library's row order (q|k|v, gate|up) and norms; the final norm."""
    layers = []
    for _ in range(g.layers):
        qk = torch.stack([d.uniform((g.head_dim,), 0.9, 1.1) / math.sqrt(g.head_dim), d.uniform((g.head_dim,), 0.9, 1.1)])
        layers.append(dict(attn_norm=d.uniform((g.dim,), 0.9, 1.1), ffn_norm=d.uniform((g.dim,), 0.9, 1.1),
                           wqkv=d.normal((g.q_width + 2 * g.kv_width, g.dim), 0.02), wo=d.normal((g.dim, g.q_width), 0.02),
                           w_gateup=d.normal((2 * g.ffn, g.dim), 0.02), wdown=d.normal((g.dim, g.ffn), 0.02),
                           qk_norms=qk, attn_scale=None, mlp_scale=None))
    return layers, d.uniform((g.dim,), 0.9, 1.1)


_PROJ = ("wqkv", "wo", "w_gateup", "wdown")


def _step_inputs(case, seed):
    """Weights, the lanes' hidden states, the caches of an ongoing generation (past positions
    filled) and the lanes' positions."""
    d, g = _Draw(seed), _stack_geometry(case)
    layers, norm = _stack_weights(d, g)
    x = d.normal((case["lanes"], g.dim))
    shape = (case["lanes"], g.n_kv, case["cap"], g.head_dim)
    dt = stack.cache_dtype(case["weight"])
    kv = [(d.normal(shape).to(dt), d.normal(shape).to(dt)) for _ in range(g.layers)]
    pos = d.ints((case["lanes"],), case["cap"] // 8, case["cap"])
    return layers, norm, x, kv, pos


def _prefill_inputs(case, seed):
    d, g = _Draw(seed), _stack_geometry(case)
    layers, norm = _stack_weights(d, g)
    x = d.normal((case["lanes"], case["t"], g.dim))
    shape = (case["lanes"], g.n_kv, case["start"], g.head_dim)
    kv = [(d.normal(shape).half(), d.normal(shape).half()) for _ in range(g.layers)]
    return layers, norm, x, kv


# ---------------------------------------------------------------- prepare and run

def _np(t):
    return t.cpu().numpy()


def _pair(p):
    return _np(p[0]), _np(p[1])


def _device_stack(g, layers, norm, weight):
    """A Stack over device weights of the kind, in its layouts."""
    def proj(w):
        if weight == "f16":
            return w.half()
        return w if weight == "f32" else ops.q8_0_repack(_q8_0(w)[0], w.shape[1])

    layers = [{k: proj(v) if k in _PROJ else v for k, v in L.items()} for L in layers]
    return stack.Stack(g, layers, norm, torch.device(DEV), weight)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "codec":
        w, latent = _codec_inputs(case, seed)
        hw = codec.HostWeights(head_w=_np(w["head"][0]), head_b=_np(w["head"][1]))
        for blk in w["blocks"]:
            hw.blocks.append(dict(act=_pair(blk["act"]), up_w=_np(blk["up"][0]), up_b=_np(blk["up"][1]), units=[
                dict(act1=_pair(u["act1"]), w1=_np(u["c1"][0]), b1=_np(u["c1"][1]), act2=_pair(u["act2"]),
                     w2=_np(u["c2"][0]), b2=_np(u["c2"][1])) for u in blk["units"]]))
        hw.out_act, (hw.out_w, hw.out_b) = _pair(w["out_act"]), _pair(w["out"])
        model = codec.Codec(codec.CONFIG5, hw, torch.device(DEV), dtype=case["dtype"])
        model.workspace(case["lanes"], case["frames"])
        latent = latent.to(model.torch_dtype)
        audio = torch.empty((case["lanes"], case["frames"] * codec.CONFIG5.hop), dtype=latent.dtype, device=DEV)
        return lambda: model.decode(latent, out=audio)
    if kind == "unit":
        i = _unit_inputs(case, seed)
        out = i["out"] if case["snake_out"] else None
        return lambda: nlc.residual_unit(i["x"], i["act1"], i["w1"], i["b1"], i["act2"], i["w2"], i["b2"], k=7,
                                         dilation=case["dilation"], snake_out=out)
    if kind == "conv":
        i = _conv_inputs(case, seed)
        return lambda: nlc.conv1d(i["x"], i["w"], i["b"], k=7, dilation=case["dilation"], snake_out=i["act"])
    if kind == "front":
        hw, codes = _front_inputs(case, seed)
        for f in vars(hw):
            v = getattr(hw, f)
            setattr(hw, f, [{k: _np(t) for k, t in e.items()} for e in v] if isinstance(v, list) else _np(v))
        model, codes = codec_front.CodecFront(codec_front.CODEC, hw, torch.device(DEV)), _np(codes).astype(np.int32)
        out = torch.empty((case["lanes"], case["frames"] * codec_front.CODEC.upsample, codec_front.CODEC.latent_dim),
                          dtype=F16, device=DEV)
        return lambda: model.decode(codes, out=out)
    g = _stack_geometry(case)
    if kind == "step":
        layers, norm, x, kv, pos = _step_inputs(case, seed)
        model = _device_stack(g, layers, norm, case["weight"])
        state = model.new_state(case["lanes"], case["cap"])
        for i, (k, v) in enumerate(kv):
            state.k[i].copy_(k)
            state.v[i].copy_(v)
        pos, out = _np(pos), torch.empty_like(x)
        return lambda: (model.decode(x, state, pos, out=out, graph=True), state.k, state.v)
    layers, norm, x, kv = _prefill_inputs(case, seed)
    model = _device_stack(g, layers, norm, "f16")
    state = model.new_state(case["lanes"], case["start"] + case["t"])
    for i, (k, v) in enumerate(kv):
        state.k[i][:, :, : case["start"]] = k
        state.v[i][:, :, : case["start"]] = v
    out = torch.empty_like(x)
    ws = torch.empty(model.prefill_workspace_bytes(case["lanes"], case["t"]), dtype=torch.uint8, device=DEV)
    return lambda: (model.prefill(x, state, case["start"], out=out, workspace=ws), state.k, state.v)


def run(state):
    return state()


# ---------------------------------------------------------------- what a pass cannot do without

def _codec_work(case):
    g, n = codec.CONFIG5, case["lanes"] * case["frames"]
    es = 2 if case["dtype"] == "f16" else 4
    params = g.channels[0] * g.latent_dim * g.head_kernel + g.channels[-1] * g.out_kernel
    for i, r in enumerate(g.rates):
        params += g.channels[i] * g.channels[i + 1] * 2 * r + 3 * 8 * g.channels[i + 1] ** 2
    return dict(bytes=es * (params + n * (g.latent_dim + g.hop)), flops=n * g.flops_per_frame())


def work(case):
    kind = case["kind"]
    if kind == "codec":
        return _codec_work(case)
    if kind in ("unit", "conv"):
        c, n, taps = case["channels"], case["lanes"] * case["length"], 8 if kind == "unit" else 7
        return dict(bytes=2 * (2 * n * c + taps * c * c), flops=2 * n * c * c * taps)
    if kind == "front":
        g, n = codec_front.CODEC, case["lanes"] * case["frames"]
        c, kvw = g.latent_dim, g.tf_n_kv * g.tf_head_dim
        params = 2 * g.book_dim * g.codebook_dim + g.codebook_dim * c * g.pre_kernel + 2 * c * g.tf_dim
        params += g.tf_layers * g.tf_dim * (2 * g.tf_heads * g.tf_head_dim + 2 * kvw + 3 * g.tf_ffn)
        params += sum(c * c * r + 8 * c * c for r in g.up_ratios)
        rows = min(n, g.book_size) * g.n_books * g.book_dim  # codebook rows looked up, f32
        return dict(bytes=2 * params + 4 * rows + n * (4 * g.n_books + 2 * g.upsample * c), flops=n * g.flops_per_frame())
    g = _stack_geometry(case)
    weights = g.weight_bytes_per_layer() // 2  # values
    if kind == "step":
        lanes, es = case["lanes"], 2 if case["weight"] == "f16" else 4
        wb = {"f16": 2.0, "f32": 4.0}.get(case["weight"], 34 / 32)
        past = (case["cap"] // 8 + case["cap"]) / 2  # a lane's positions, on average
        kv = 2 * lanes * past * g.kv_width
        return dict(bytes=g.layers * (wb * weights + es * kv) + 8 * lanes * g.dim,
                    flops=g.layers * lanes * (2 * weights + 4 * past * g.q_width))
    rows = case["lanes"] * case["t"]
    keys = case["start"] + (case["t"] + 1) / 2
    kv = 2 * case["lanes"] * (case["start"] + case["t"]) * g.kv_width
    return dict(bytes=g.layers * 2 * (weights + kv) + 8 * rows * g.dim,
                flops=g.layers * rows * (2 * weights + 4 * keys * g.q_width))


def tolerance(case):
    """About four times what the path is measured to be off ``exact``: f16 storage (or Q8_0
    activation codes) where the path has it, f32 sums elsewhere."""
    kind = case["kind"]
    if kind == "codec":  # f16: rounding at every stored activation, carried through 24 SnakeBetas
        return {"rel": 1.3e-2} if case["dtype"] == "f16" else {"rel": 4e-5}
    if kind in ("unit", "conv"):
        return {"rel": 1.8e-3 if kind == "unit" else 1.2e-3}
    if kind == "front":
        return {"rel": 4.5e-3}
    if kind == "step":  # q8_0: an activation at a code's boundary may take the other code
        return {"rel": {"f16": 1.6e-3, "q8_0": 2e-2}.get(case["weight"], 4e-6)}
    return {"rel": 2e-3}


# ---------------------------------------------------------------- float64

def _snake64(x, act):
    a, r = act[0].to(F64), act[1].to(F64)
    return x + r * torch.sin(a * x) ** 2


def _conv64(x, w, b, dilation=1):
    """Causal channels-last conv: x [lanes, L, cin], w [cout, cin, k]."""
    k, length = w.shape[2], x.shape[1]
    y = torch.empty((x.shape[0], length, w.shape[0]), dtype=F64, device=x.device)
    taps = [w[:, :, t].to(F64).t().contiguous() for t in range(k)]
    for i in range(x.shape[0]):
        y[i] = x[i] @ taps[k - 1]
        for t in range(k - 1):
            off = (k - 1 - t) * dilation
            if off < length:
                y[i, off:] += x[i, : length - off] @ taps[t]
    return y if b is None else y + b.to(F64)


def _taps_last(w, c):
    """A tap-major weight [cout, k * cin] as [cout, cin, k]."""
    return w.view(w.shape[0], -1, c).transpose(1, 2)


def _unit64(x, act1, w1, b1, act2, w2, b2, dilation):
    h = _conv64(_snake64(x, act1), w1, b1, dilation)
    return x + _conv64(_snake64(h, act2), w2, b2)


def _up64(x, w, b, rate):
    """ConvTranspose1d [cin, cout, k], stride rate, the trailing k - rate outputs dropped."""
    lanes, length, _ = x.shape
    cout, k = w.shape[1], w.shape[2]
    y = torch.zeros((lanes, length, rate, cout), dtype=F64, device=x.device)
    for t in range(k):
        j, p = divmod(t, rate)
        v = torch.stack([xi @ w[:, :, t].to(F64) for xi in x])
        y[:, j:, p] += v[:, : length - j]
    return y.view(lanes, length * rate, cout) + b.to(F64)


def _exact_codec(case, seed):
    w, latent = _codec_inputs(case, seed)
    dt, g = F16 if case["dtype"] == "f16" else F32, codec.CONFIG5

    def cw(p):  # weights and biases as the codec holds them
        return p[0].to(dt), p[1].to(dt)

    x = _conv64(latent.to(dt).to(F64), *cw(w["head"]))
    for i, blk in enumerate(w["blocks"]):
        x = _up64(_snake64(x, blk["act"]), *cw(blk["up"]), g.rates[i])
        for u, dil in zip(blk["units"], g.ru_dilations):
            x = _unit64(x, u["act1"], *cw(u["c1"]), u["act2"], *cw(u["c2"]), dil)
    return torch.tanh(_conv64(_snake64(x, w["out_act"]), *cw(w["out"])))[..., 0]


def _rms64(x, gamma, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gamma.to(F64)


def _rope64(x, pos, base):
    """Half-split RoPE of x [..., n, D] at positions pos [n] (or broadcastable [..., n])."""
    half = x.shape[-1] // 2
    freq = base ** (-2.0 * torch.arange(half, dtype=F64, device=x.device) / x.shape[-1])
    ph = pos.to(F64)[..., None] * freq
    c, s = torch.cos(ph), torch.sin(ph)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _exact_front(case, seed):
    hw, codes = _front_inputs(case, seed)
    g = codec_front.CODEC

    def lin(x, w, b=None):
        y = x @ w.half().to(F64).t()
        return y if b is None else y + b.half().to(F64)

    pick = [hw.codebooks[i][codes[..., i]].to(F64) for i in range(g.n_books)]
    q = lin(sum(pick[: g.n_first]), hw.out_proj_sem[..., 0]) + lin(sum(pick[g.n_first:]), hw.out_proj_ac[..., 0])
    h = lin(_conv64(q, hw.pre_w.half(), hw.pre_b.half()), hw.in_w, hw.in_b)
    lanes, t, hd = h.shape[0], h.shape[1], g.tf_head_dim
    pos = torch.arange(t, device=DEV)
    seen = (pos[None] <= pos[:, None]) & (pos[None] > pos[:, None] - g.tf_window)

    def heads(x, n):
        return x.view(lanes, t, n, hd).transpose(1, 2)

    for L in hw.layers:
        a = _rms64(h, L["attn_norm"], g.tf_eps)
        q = _rope64(heads(lin(a, L["wq"]), g.tf_heads), pos, g.tf_rope_base)
        k = _rope64(heads(lin(a, L["wk"]), g.tf_n_kv), pos, g.tf_rope_base)
        v = heads(lin(a, L["wv"]), g.tf_n_kv)
        s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(hd)
        o = torch.matmul(torch.softmax(s.masked_fill(~seen, -math.inf), -1), v.contiguous())
        h = h + lin(o.transpose(1, 2).reshape(lanes, t, -1), L["wo"]) * L["attn_scale"].to(F64)
        a = _rms64(h, L["ffn_norm"], g.tf_eps)
        m = torch.nn.functional.silu(lin(a, L["gate"])) * lin(a, L["up"])
        h = h + lin(m, L["down"]) * L["mlp_scale"].to(F64)
    x = lin(_rms64(h, hw.tf_norm, g.tf_eps), hw.out_w, hw.out_b)
    for U, r in zip(hw.up, g.up_ratios):
        u = _up64(x, U["up_w"].half(), U["up_b"].half(), r)
        dn = sum(torch.nn.functional.pad(u, (0, 0, g.dw_kernel - 1 - i, 0))[:, : u.shape[1]] * U["dw_w"][:, 0, i].to(F64)
                 for i in range(g.dw_kernel)) + U["dw_b"].to(F64)
        dn = torch.nn.functional.layer_norm(dn, (dn.shape[-1],), U["ln_w"].to(F64), U["ln_b"].to(F64), g.ln_eps)
        p = torch.nn.functional.gelu(lin(dn, U["pw1_w"], U["pw1_b"]))
        x = u + lin(p, U["pw2_w"], U["pw2_b"]) * U["gamma"].to(F64)
    return x


def _weights64(layers, weight):
    def proj(w):
        if weight in ("q8_0", "q8_0_a32"):
            return _q8_0(w)[1]
        return (w.half() if weight == "f16" else w).to(F64)

    return [{k: proj(v) if k in _PROJ else v for k, v in L.items()} for L in layers]


def _mlp64(h, L, g):
    gate, up = (_rms64(h, L["ffn_norm"], g.eps) @ L["w_gateup"].t()).split(g.ffn, -1)
    return h + (torch.nn.functional.silu(gate) * up) @ L["wdown"].t()


def _qkv64(h, L, g):
    """Normed, roped-to-be q, k and v of rows h [..., dim] as [..., heads, D]."""
    qkv = (_rms64(h, L["attn_norm"], g.eps) @ L["wqkv"].t()).view(*h.shape[:-1], g.heads + 2 * g.n_kv, g.head_dim)
    q, k, v = qkv.split([g.heads, g.n_kv, g.n_kv], -2)
    return _rms64(q, L["qk_norms"][0], g.eps), _rms64(k, L["qk_norms"][1], g.eps), v


def _exact_step(case, seed):
    g = _stack_geometry(case)
    layers, norm, x, kv, pos = _step_inputs(case, seed)
    lanes, h, ks, vs = case["lanes"], x.to(F64), [], []
    lane = torch.arange(lanes, device=DEV)
    seen = torch.arange(case["cap"], device=DEV)[None] <= pos[:, None]
    for L, (kc, vc) in zip(_weights64(layers, case["weight"]), kv):
        q, k, v = _qkv64(h, L, g)
        q, k = _rope64(q, pos[:, None], g.rope_base), _rope64(k, pos[:, None], g.rope_base)
        kc, vc = kc.to(F64), vc.to(F64)
        kc[lane, :, pos], vc[lane, :, pos] = k, v
        o = torch.empty((lanes, g.n_kv, g.gqa, g.head_dim), dtype=F64, device=DEV)
        for i in range(lanes):
            s = torch.matmul(q[i].view(g.n_kv, g.gqa, -1), kc[i].transpose(1, 2).contiguous())
            o[i] = torch.matmul(torch.softmax(s.masked_fill(~seen[i], -math.inf), -1), vc[i])
        h = _mlp64(h + o.view(lanes, -1) @ L["wo"].t(), L, g)
        ks.append(kc)
        vs.append(vc)
    return _rms64(h, norm, g.eps), ks, vs


def _exact_prefill(case, seed):
    g = _stack_geometry(case)
    layers, norm, x, kv = _prefill_inputs(case, seed)
    h, ks, vs, start, t = x.to(F64), [], [], case["start"], case["t"]
    pos = start + torch.arange(t, device=DEV)
    seen = torch.arange(start + t, device=DEV)[None] <= pos[:, None]
    for L, (kc, vc) in zip(_weights64(layers, "f16"), kv):
        q, k, v = _qkv64(h, L, g)
        q, k = (_rope64(a.transpose(1, 2).contiguous(), pos, g.rope_base) for a in (q, k))
        kc, vc = torch.cat([kc.to(F64), k], 2), torch.cat([vc.to(F64), v.transpose(1, 2)], 2)
        o = torch.empty((case["lanes"], t, g.heads, g.head_dim), dtype=F64, device=DEV)
        for i in range(case["lanes"]):
            for j in range(g.heads):
                s = q[i, j] @ kc[i, j // g.gqa].t().contiguous()
                o[i, :, j] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ vc[i, j // g.gqa]
        h = _mlp64(h + o.view(*h.shape[:-1], -1) @ L["wo"].t(), L, g)
        ks.append(kc)
        vs.append(vc)
    return _rms64(h, norm, g.eps), ks, vs


def exact(case, seed):
    kind = case["kind"]
    if kind == "codec":
        return _exact_codec(case, seed)
    if kind == "unit":
        i, c = _unit_inputs(case, seed), case["channels"]
        y = _unit64(i["x"].to(F64), i["act1"], _taps_last(i["w1"], c), i["b1"], i["act2"], _taps_last(i["w2"], c), i["b2"],
                    case["dilation"])
        return _snake64(y, i["out"]) if case["snake_out"] else y
    if kind == "conv":
        i = _conv_inputs(case, seed)
        return _snake64(_conv64(i["x"].to(F64), _taps_last(i["w"], case["channels"]), i["b"], case["dilation"]), i["act"])
    if kind == "front":
        return _exact_front(case, seed)
    return _exact_step(case, seed) if kind == "step" else _exact_prefill(case, seed)
