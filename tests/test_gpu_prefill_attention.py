"""The prefill's 32-query attention blocks at their edges, against the oracle with the prefill's bars
(outputs 5e-4, written cache entries 1e-3): query counts around a block, key ranges that end inside a
32-key block of either kind (the cache's rows, the new ones), windows that mask whole blocks for some
of a block's queries, few and many workgroups. Fewer than 16 queries run on the per-wave kernel, whose
scores in LDS set its queries per wave and waves per workgroup by the number of keys."""
from dataclasses import replace

import pytest
import torch

import oracle
from dtts import stack, synth

from _stack_ref import SMALL, WINDOWED, inputs
from _util import rel, to_dev, to_host

pytestmark = pytest.mark.gpu

LONG = replace(SMALL, layers=1, capacity=1024)
DEEP = replace(LONG, capacity=8200)
WIN = replace(WINDOWED, layers=1, window=40, capacity=1024)


@pytest.mark.parametrize("geo,lanes,t,start", [
    (LONG, 1, 16, 0), (LONG, 2, 31, 1), (LONG, 1, 32, 31), (LONG, 2, 33, 32), (LONG, 1, 65, 33), (LONG, 1, 129, 700),
    (LONG, 1, 500, 0), (WIN, 1, 16, 0), (WIN, 2, 45, 39), (WIN, 1, 100, 41), (WIN, 1, 300, 500), (LONG, 40, 200, 5),
    # the per-wave kernel: key ranges past one and several strides of 64 lanes, four waves a workgroup (up to
    # 896 keys), two (up to 1920) and one; four queries a wave (up to 3968 keys), two and one
    (LONG, 2, 2, 60), (LONG, 1, 3, 64), (LONG, 3, 5, 500), (LONG, 1, 15, 900), (LONG, 2, 2, 127), (WIN, 2, 9, 500),
    (DEEP, 1, 15, 2000), (DEEP, 1, 6, 4000), (DEEP, 1, 3, 8100),
])
def test_prefill_attention_blocks(dev, geo, lanes, t, start):
    layers, fn = stack.random_weights(geo, 7)
    cap = start + t
    _, kc, vc = inputs(geo, 7, lanes, cap)
    x = synth.normal(7, "prefill.x", (lanes, t, geo.dim))
    st = stack.Stack(geo, layers, fn, dev)
    state = st.new_state(lanes, cap)
    state.k[0].copy_(to_dev(kc[0], dev))
    state.v[0].copy_(to_dev(vc[0], dev))
    want = oracle.stack_prefill_f32(geo, layers, fn, x, kc, vc, start)
    got = to_host(st.prefill(to_dev(x, dev), state, start))
    torch.cuda.synchronize()
    assert rel(got, want)[1] < 5e-4, rel(got, want)
    for g, w in ((state.k[0], kc[0]), (state.v[0], vc[0])):
        assert rel(synth.from_f16_bits(to_host(g)), synth.from_f16_bits(w))[1] < 1e-3


@pytest.mark.parametrize("geo,lanes,t,start", [(LONG, 40, 200, 5), (LONG, 3, 300, 40), (WIN, 70, 129, 0)])
def test_prompt_alone_and_in_a_batch(dev, geo, lanes, t, start):
    """A prompt of more than 128 positions gives the same bits alone and beside others, whether or not
    the batch fills the chip."""
    layers, fn = stack.random_weights(geo, 8)
    _, kc, vc = inputs(geo, 8, lanes, start + t)
    st = stack.Stack(geo, layers, fn, dev)
    x = to_dev(synth.normal(8, "prefill.x", (lanes, t, geo.dim)), dev)
    outs = []
    for sl in (slice(0, lanes), slice(lanes - 1, lanes)):
        state = st.new_state(sl.stop - sl.start, start + t)
        state.k[0].copy_(to_dev(kc[0][sl], dev))
        state.v[0].copy_(to_dev(vc[0][sl], dev))
        outs.append((st.prefill(x[sl].contiguous(), state, start), state.k[0], state.v[0]))
    for batch, alone in zip(*outs):
        assert torch.equal(batch[-1], alone[0])


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("geo,lanes,t,start,at", [
    (LONG, 1, 500, 0, 490), (LONG, 2, 100, 40, 33), (LONG, 1, 600, 300, 599), (LONG, 1, 20, 0, 19), (WIN, 1, 300, 500, 170),
])
def test_non_finite_position_stays_with_the_queries_that_see_it(dev, geo, lanes, t, start, at, value):
    """A new position that is not finite leaves every earlier query's output as it is, and every query past
    its window: its value is never multiplied into a query that does not see it."""
    layers, fn = stack.random_weights(geo, 9)
    _, kc, vc = inputs(geo, 9, lanes, start + t)
    st = stack.Stack(geo, layers, fn, dev)
    x = to_dev(synth.normal(9, "prefill.x", (lanes, t, geo.dim)), dev)

    def run(x):
        state = st.new_state(lanes, start + t)
        state.k[0].copy_(to_dev(kc[0], dev))
        state.v[0].copy_(to_dev(vc[0], dev))
        return st.prefill(x, state, start)

    want = run(x)
    x[lanes - 1, at] = value
    got = run(x)
    seen = torch.zeros((lanes, t), dtype=torch.bool, device=dev)
    seen[lanes - 1, at:min(t, at + geo.window) if geo.window else t] = True
    assert torch.isfinite(got[~seen]).all()
    assert rel(to_host(got[~seen]), to_host(want[~seen]))[1] < 5e-4
    assert torch.isnan(got[seen]).all()


def test_non_finite_cache_value_past_the_window(dev):
    """An infinite cached value reaches the queries whose window holds it and no other of their block."""
    layers, fn = stack.random_weights(WIN, 10)
    t, start, at = 70, 90, 60  # seen by queries up to position 99, ti 9
    _, kc, vc = inputs(WIN, 10, 1, start + t)
    st = stack.Stack(WIN, layers, fn, dev)
    x = to_dev(synth.normal(10, "prefill.x", (1, t, WIN.dim)), dev)
    outs = []
    for value in (None, float("inf")):
        state = st.new_state(1, start + t)
        state.k[0].copy_(to_dev(kc[0], dev))
        state.v[0].copy_(to_dev(vc[0], dev))
        if value:
            state.v[0][0, :, at] = value
        outs.append(st.prefill(x, state, start)[0])
    seen = at + WIN.window - start
    assert not torch.isfinite(outs[1][:seen]).any()
    assert rel(to_host(outs[1][seen:]), to_host(outs[0][seen:]))[1] < 5e-4
