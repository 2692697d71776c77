"""dtts_stack_decode (one decode step of a Qwen3 decoder stack, Stack::forward at t = 1,
crates/qwen3tts/src/qwen3.rs:294-467) against the oracle's restatement on the same seeded
weights, inputs and cache history: the normed output within max-rel 2e-4 (f32 sums in another
order; an f16 activation rounding may flip), every cache entry written at a lane's position
within max-rel 1e-3 (qkrope.rs's own bar for cached f16) and every other entry bit-identical.
Eager launches and the captured graph run the same kernels and must agree bit for bit, step
after step as positions advance. Geometries: QK-norm (talker / code predictor form) and
no-QK-norm with LayerScale and a sliding window (the codec transformer's form), caches long
enough for the attention split, the talker's own widths, and the argument checks."""
import ctypes
from dataclasses import replace

import numpy as np
import pytest
import torch

import oracle
from dtts import DttsError, stack, synth
from dtts._lib import call

from _stack_ref import SMALL, WINDOWED, inputs, with_layers
from _util import rel, to_dev, to_host

pytestmark = pytest.mark.gpu


class Pair:
    """The GPU stack and the oracle on the same weights and cache history."""

    def __init__(self, dev, geo, seed, lanes, cap, tol=2e-4):
        self.geo, self.lanes, self.cap, self.tol = geo, lanes, cap, tol
        self.layers, self.fn = stack.random_weights(geo, seed)
        self.x, self.kc, self.vc = inputs(geo, seed, lanes, cap)
        self.st = stack.Stack(geo, self.layers, self.fn, dev)
        self.state = self.st.new_state(lanes, cap)
        for i in range(geo.layers):
            self.state.k[i].copy_(to_dev(self.kc[i], dev))
            self.state.v[i].copy_(to_dev(self.vc[i], dev))
        self.dev = dev

    def step(self, pos, scale=1.0, graph=False, out=None):
        xs = (self.x * np.float32(scale)).astype(np.float32)
        before = [(k.copy(), v.copy()) for k, v in zip(self.kc, self.vc)]
        want = oracle.stack_decode_f32(self.geo, self.layers, self.fn, xs, self.kc, self.vc, pos)
        xd = to_dev(xs, self.dev) if out is None else out[0]
        if out is not None:
            xd.copy_(torch.from_numpy(xs))
        got = self.st.decode(xd, self.state, pos, graph=graph, out=None if out is None else out[1])
        torch.cuda.synchronize()
        got = to_host(got)
        assert rel(got, want)[1] < self.tol, rel(got, want)
        pos = np.broadcast_to(np.asarray(pos), (self.lanes,))
        for li in range(self.geo.layers):
            for dev_t, ora, old in ((self.state.k[li], self.kc[li], before[li][0]),
                                    (self.state.v[li], self.vc[li], before[li][1])):
                g = to_host(dev_t)
                mask = np.ones(g.shape, bool)
                for i, p in enumerate(pos):
                    mask[i, :, p] = False
                assert np.array_equal(g[mask], old[mask]), "a cache slot off the lanes' positions changed"
                assert rel(synth.from_f16_bits(g[~mask]), synth.from_f16_bits(ora[~mask]))[1] < 1e-3
                # continue from the GPU's own cache so both sides share one history
                ora[...] = g
        return got


def test_stack_step_matches_oracle(dev):
    p = Pair(dev, SMALL, 90, 5, 64)
    p.step(np.array([0, 63, 17, 40, 1], np.int32))


@pytest.mark.parametrize("lanes", [1, 8, 16, 9])
def test_stack_routes_projections_by_lane_count(dev, lanes):
    """Proj::Half's routing (crates/tts-nn/src/lib.rs:516-529, skinny.rs:123-131): 8 and 16 lanes
    keep the skinny GEMM's f32 outputs; 1 lane (a single utterance's decode) and 9 take candle's
    f16 matmul, whose outputs are f16 -- on the graph path too."""
    p = Pair(dev, SMALL, 95, lanes, 64)
    start = synth.randint(95, "stack.route.pos", (lanes,), 0, 60).astype(np.int32)
    p.step(start)
    p.step(start + 1, graph=True)


def test_stack_steps_advance_eager_and_graph_agree(dev):
    """Three steps eager, then the same three steps again from the same history as a graph."""
    lanes, cap = 6, 64
    start = np.array([0, 5, 60, 30, 11, 2], np.int32)
    a = Pair(dev, SMALL, 91, lanes, cap)
    b = Pair(dev, SMALL, 91, lanes, cap)
    xo = (torch.empty((lanes, SMALL.dim), device=dev), torch.empty((lanes, SMALL.dim), device=dev))
    for s in range(3):
        ea = a.step(start + s, scale=1 + 0.2 * s)
        gb = b.step(start + s, scale=1 + 0.2 * s, graph=True, out=xo)
        assert np.array_equal(ea, gb), f"graph replay differs from eager at step {s}"
    for i in range(SMALL.layers):
        assert torch.equal(a.state.k[i], b.state.k[i]) and torch.equal(a.state.v[i], b.state.v[i])


def test_stack_windowed_layer_scale_no_qk_norm(dev):
    p = Pair(dev, WINDOWED, 92, 4, 32)
    start = np.array([0, 3, 20, 27], np.int32)
    for s in range(4):
        p.step(start + s, scale=1 + 0.1 * s, graph=(s % 2 == 1))


def test_stack_long_cache_splits_attention(dev):
    """cap 700: chunks of 128 positions merged by a second launch."""
    geo = replace(SMALL, capacity=700)
    p = Pair(dev, geo, 93, 4, 700)
    p.step(np.array([699, 256, 0, 513], np.int32))
    p.step(np.array([699, 257, 1, 514], np.int32) - np.array([1, 0, 0, 0], np.int32), graph=True)


def test_stack_talker_widths(dev):
    """The talker's own widths (dim 2048, 16/8 heads, D 128, ffn 6144), 2 of its 28 layers,
    48 lanes (the configs' batch) at per-lane positions. Bar 1e-3: at these widths f16
    activation roundings that land on the other side of a tie already separate the oracle from
    a float64 evaluation of the same step by max-rel 3.0e-4 (seed 94)."""
    geo = with_layers(replace(stack.TALKER, capacity=256), 2)
    lanes = 48
    p = Pair(dev, geo, 94, lanes, 256, tol=1e-3)
    p.step(synth.randint(94, "stack.talker.pos", (lanes,), 0, 255).astype(np.int32), graph=True)


def test_stack_talker_long_cache_graph_replays(dev):
    """The talker's widths at a cache capacity of 2048: 1 to 16 chunks of 128 per (lane, kv head), spans
    ending on and either side of chunk boundaries; an eager step, then graph replays as the
    positions advance."""
    geo = with_layers(replace(stack.TALKER, capacity=2048), 2)
    lanes = 8
    p = Pair(dev, geo, 97, lanes, 2048, tol=1e-3)
    start = np.array([2040, 1535, 1536, 511, 512, 1024, 7, 1900], np.int32)
    for s in range(4):
        p.step(start + s, graph=(s > 0))


def test_stack_rejects_bad_arguments(dev):
    geo = SMALL
    layers, fn = stack.random_weights(geo, 95)
    st = stack.Stack(geo, layers, fn, dev)
    state = st.new_state(3, 16)
    x = torch.zeros((3, geo.dim), device=dev)
    with pytest.raises(DttsError, match="exceeds cache capacity"):
        st.decode(x, state, np.array([0, 16, 2], np.int32))
    with pytest.raises(DttsError, match="capacity"):
        st.decode(x, st.new_state(3, 65), 0)  # cache longer than the RoPE table
    big = st.new_state(65, 4)
    with pytest.raises(DttsError, match="lanes"):
        st.decode(torch.zeros((65, geo.dim), device=dev), big, 0, workspace=torch.empty(16, dtype=torch.uint8, device=dev))
    with pytest.raises(DttsError, match="workspace"):
        st.decode(x, state, 0, workspace=torch.empty(256, dtype=torch.uint8, device=dev))
    torch.cuda.synchronize()
    for t in state.k + state.v:
        assert not t.any(), "a rejected call wrote the cache"
    with pytest.raises(DttsError, match="heads"):
        stack.Stack(replace(geo, heads=3), layers, fn, dev)
    with pytest.raises(DttsError, match="multiples of 128"):
        stack.Stack(replace(geo, ffn=500), stack.random_weights(replace(geo, ffn=500), 95)[0], fn, dev)


# ---------------------------------------------------------------- f32 and Q8_0 layers
# Stack::load with Weight::F32 or Weight::Quant (crates/qwen3tts/src/qwen3.rs:228-250): f32
# caches, Proj::forward's f32 activations into every projection (lib.rs:509-531), the composed QK
# route. Bars against oracle.stack_decode_f32(weight=...): f32 and the unquantized-activation Q8_0
# kind max-rel 1e-5 on the output and on every cache entry written (f32 sums in another order);
# W8A8 2e-2, the north star's tolerance for int8 GEMM outputs at unit scale: an activation whose
# f32 value differs from the oracle's in the last bit can land on the other side of a code's
# rounding boundary (one code step of one block moves a dot by ~4/(127 sqrt(k)) of it), and the
# next projections then quantize shifted inputs, so GPU and oracle become two W8A8 evaluations
# apart by the quantization noise itself (measured: 1e-7 until a first flip, 6e-4 after one at the
# small widths, 7.7e-3 at the talker's; the per-projection W8A8 kernel is held to 1e-5 on
# identical inputs in test_gpu_gemm.py); every other cache entry bit-identical.

class PairW(Pair):
    def __init__(self, dev, geo, seed, lanes, cap, weight, tol):
        self.geo, self.lanes, self.cap, self.tol, self.weight = geo, lanes, cap, tol, weight
        self.layers, self.fn = stack.random_weights(geo, seed)
        self.x, self.kc, self.vc = inputs(geo, seed, lanes, cap, weight=weight)
        self.st = stack.Stack(geo, self.layers, self.fn, dev, weight=weight)
        self.state = self.st.new_state(lanes, cap)
        assert self.state.k[0].dtype == torch.float32
        for i in range(geo.layers):
            self.state.k[i].copy_(torch.from_numpy(self.kc[i]).to(dev))
            self.state.v[i].copy_(torch.from_numpy(self.vc[i]).to(dev))
        self.dev = dev

    def step(self, pos, scale=1.0, graph=False):
        xs = (self.x * np.float32(scale)).astype(np.float32)
        before = [(k.copy(), v.copy()) for k, v in zip(self.kc, self.vc)]
        want = oracle.stack_decode_f32(self.geo, self.layers, self.fn, xs, self.kc, self.vc, pos, weight=self.weight)
        got = to_host(self.st.decode(to_dev(xs, self.dev), self.state, pos, graph=graph))
        torch.cuda.synchronize()
        worst = rel(got, want)[1]
        assert worst < self.tol, (self.weight, worst)
        pos = np.broadcast_to(np.asarray(pos), (self.lanes,))
        for li in range(self.geo.layers):
            for dev_t, ora, old in ((self.state.k[li], self.kc[li], before[li][0]),
                                    (self.state.v[li], self.vc[li], before[li][1])):
                g = to_host(dev_t)
                mask = np.ones(g.shape, bool)
                for i, p in enumerate(pos):
                    mask[i, :, p] = False
                assert np.array_equal(g[mask], old[mask]), "a cache slot off the lanes' positions changed"
                worst_c = rel(g[~mask], ora[~mask])[1]
                assert worst_c < self.tol, (self.weight, "cache", worst_c)
                ora[...] = g
        print(f"{self.weight}: out max-rel {worst:.2e}", flush=True)
        return got


KIND_TOL = {"f32": 1e-5, "q8_0_a32": 1e-5, "q8_0": 2e-2}


@pytest.mark.parametrize("weight", ["f32", "q8_0", "q8_0_a32"])
def test_stack_weight_kinds_small(dev, weight):
    """QK-norm geometry and the windowed, LayerScale, no-QK-norm one, steps eager and graph."""
    p = PairW(dev, replace(SMALL, dim=256, ffn=512), 96, 5, 64, weight, KIND_TOL[weight])
    start = np.array([0, 63, 17, 40, 1], np.int32) - np.array([0, 2, 0, 0, 0], np.int32)
    p.step(start)
    p.step(start + 1, graph=True)
    w = PairW(dev, replace(WINDOWED, dim=256, ffn=512, heads=4, n_kv=4), 97, 4, 32, weight, KIND_TOL[weight])
    pos = np.array([0, 3, 20, 27], np.int32)
    for s in range(3):
        w.step(pos + s, scale=1 + 0.1 * s, graph=(s % 2 == 1))


@pytest.mark.parametrize("weight", ["f32", "q8_0", "q8_0_a32"])
def test_stack_weight_kinds_talker_widths(dev, weight):
    """The talker's widths (dim 2048, 16/8 heads, D 128, ffn 6144), 2 of its 28 layers, 48 lanes
    at per-lane positions, through the captured graph."""
    geo = with_layers(replace(stack.TALKER, capacity=256), 2)
    lanes = 48
    p = PairW(dev, geo, 98, lanes, 256, weight, KIND_TOL[weight])
    p.step(synth.randint(98, "stack.talker.pos", (lanes,), 0, 254).astype(np.int32), graph=True)


def test_stack_weight_kind_checks(dev):
    """Q8_0 layers need widths that are multiples of 256 (the packed layout); the prefill branch
    runs f16 stacks only; an unknown kind is refused."""
    geo = replace(SMALL, dim=256, ffn=640)
    layers, fn = stack.random_weights(geo, 99)
    with pytest.raises(DttsError, match="multiples? of 256"):  # the repack at upload, or create itself
        stack.Stack(geo, layers, fn, dev, weight="q8_0")
    # create's own check, on weights whose rows the repack accepted
    geo_ok = replace(SMALL, dim=256, ffn=512)
    ok = stack.Stack(geo_ok, *stack.random_weights(geo_ok, 99), dev, weight="q8_0")
    g = stack.c_geometry(replace(geo_ok, ffn=640))
    handle = ctypes.c_void_p()
    with pytest.raises(DttsError, match="multiples of 256"):
        call("dtts_stack_create_as", ctypes.byref(g), ctypes.cast(ok._l, ctypes.c_void_p),
             ctypes.c_void_p(ok._keep[0].data_ptr()), stack.WEIGHTS["q8_0"], ctypes.byref(handle))
    geo = SMALL
    layers, fn = stack.random_weights(geo, 99)
    st = stack.Stack(geo, layers, fn, dev, weight="f32")
    with pytest.raises(DttsError, match="f16 layers"):
        st.prefill(torch.zeros((1, 2, geo.dim), device=dev), st.new_state(1, 16), 0,
                   workspace=torch.empty(256, dtype=torch.uint8, device=dev))
    stack.WEIGHTS["bogus"] = 7
    try:
        with pytest.raises(DttsError, match="weight kind 7"):
            stack.Stack(geo, layers, fn, dev, weight="bogus")
    finally:
        del stack.WEIGHTS["bogus"]
