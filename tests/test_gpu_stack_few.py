"""The decode step at few lanes against the oracle, where its attention splits spans into shorter chunks:
positions on both sides of a chunk's edge, one lane to the batch that fills the chip, both cache types,
grouped heads and windows, on both sides of the lines to which the attention makes its own q, k and v
(128 (lane, kv head) pairs, or two chunks; up to four query heads per kv head). Bars as test_gpu_stack.py's."""
from dataclasses import replace

import numpy as np
import pytest
import torch

import oracle
from dtts import stack, synth

from _stack_ref import SMALL, WINDOWED, inputs
from _util import rel, to_dev, to_host

pytestmark = pytest.mark.gpu

ONE = replace(SMALL, layers=1, capacity=1600)
EIGHT = replace(SMALL, layers=1, heads=8, n_kv=8, head_dim=64, capacity=1600)


def edges(lanes, cap, chunk):
    """A position per lane: both sides of every chunk's edge, the first and the last, in turn."""
    at = sorted({p for e in range(0, cap + chunk, chunk) for p in (e - 1, e, e + 1) if 0 <= p < cap} | {cap - 1})
    return [at[(i * 5) % len(at)] for i in range(lanes)]



@pytest.mark.parametrize("geo,weight,lanes,cap,pos", [
    (ONE, "f16", 1, 256, [255]),                      # one chunk
    (ONE, "f16", 1, 257, [256]), (ONE, "f16", 1, 320, [319]),  # still one
    (ONE, "f16", 1, 321, [320]), (ONE, "f32", 1, 257, [256]),  # three of 128, the last of 65 and of one position
    (ONE, "f16", 1, 385, [384]),                      # four, the last of one
    (ONE, "f16", 3, 700, [0, 127, 128]),
    (ONE, "f16", 8, 1600, [0, 1, 255, 256, 511, 512, 1023, 1599]),
    (ONE, "f16", 50, 300, [(i * 37) % 300 for i in range(50)]),
    # seventeen and thirty-three chunks of 128: the merge in two and three rounds
    (replace(ONE, capacity=4200), "f16", 2, 4100, [4099, 2048]), (replace(ONE, capacity=4200), "f32", 1, 2049, [2048]),
    (ONE, "q8_0_a32", 2, 1500, [1499, 128]),
    (ONE, "f32", 9, 520, [0, 63, 64, 127, 128, 129, 384, 511, 519]),
    (replace(ONE, n_kv=4), "f16", 2, 400, [399, 200]),  # one query head per kv head
    (replace(ONE, heads=8, n_kv=1, head_dim=64), "f16", 2, 400, [399, 129]),  # eight
    (replace(ONE, heads=8, n_kv=1), "f32", 3, 700, [699, 384, 5]), (replace(ONE, heads=8, n_kv=1), "f16", 2, 64, [63, 0]),
    # four: in the attention's launch from two chunks on
    (replace(ONE, heads=8), "f16", 2, 64, [63, 0]), (replace(ONE, heads=8), "f16", 3, 700, [699, 384, 5]),
    (replace(ONE, heads=8, head_dim=64), "f32", 3, 1500, [1499, 128, 127]), (replace(ONE, heads=8), "f32", 2, 200, [199, 1]),
    (replace(WINDOWED, layers=1, window=300, capacity=700), "f16", 4, 700, [10, 299, 300, 699]),
    (replace(WINDOWED, layers=1, window=400, capacity=700), "f16", 4, 700, [10, 399, 400, 699]),
    # more than 128 pairs: three chunks or more after the qk-rope kernel, up to two without it
    (replace(EIGHT, heads=16), "f16", 17, 1100, edges(17, 1100, 128)), (EIGHT, "f32", 17, 1100, edges(17, 1100, 128)),
    (EIGHT, "f16", 17, 1100, edges(17, 1100, 256)), (EIGHT, "f32", 33, 600, edges(33, 600, 256)),
    (EIGHT, "f16", 48, 1536, edges(48, 1536, 512)), (EIGHT, "f32", 48, 1025, edges(48, 1025, 512)),
    (replace(EIGHT, heads=16, head_dim=128), "f16", 24, 1100, edges(24, 1100, 256)),
    (replace(WINDOWED, layers=1, heads=8, n_kv=8, window=700, capacity=1100), "f16", 24, 1100, edges(24, 1100, 256)),
    (EIGHT, "f16", 48, 1000, edges(48, 1000, 512)), (EIGHT, "f32", 49, 257, edges(49, 257, 256)),
    # (a multiple of 8 lanes: at 17 a projection's sum near a midpoint of its f16 rounding, 1.0959 against
    # 1.0949, is one ulp of 2^-10 off, 2.7e-4 of the largest output, on either side of the line alike)
    (replace(EIGHT, heads=16, head_dim=128), "f16", 24, 17, edges(24, 17, 16)),
])
def test_step_few_lanes(dev, geo, weight, lanes, cap, pos):
    layers, fn = stack.random_weights(geo, 11)
    x, kc, vc = inputs(geo, 11, lanes, cap, weight=weight)
    st = stack.Stack(geo, layers, fn, dev, weight)
    state = st.new_state(lanes, cap)
    put = to_dev if weight == "f16" else lambda a, d: torch.from_numpy(a).to(d)
    state.k[0].copy_(put(kc[0], dev))
    state.v[0].copy_(put(vc[0], dev))
    pos = np.asarray(pos, np.int32)
    want = oracle.stack_decode_f32(geo, layers, fn, x, kc, vc, pos, weight)
    got = to_host(st.decode(to_dev(x, dev), state, pos))
    torch.cuda.synchronize()
    bar = 2e-4 if weight == "f16" else 1e-5
    assert rel(got, want)[1] < bar, rel(got, want)
    back = synth.from_f16_bits if weight == "f16" else np.asarray
    for g, w in ((state.k[0], kc[0]), (state.v[0], vc[0])):
        g = to_host(g) if weight == "f16" else g.cpu().numpy()
        for i, p in enumerate(pos):
            off = np.arange(cap) != p
            assert np.array_equal(g[i][:, off], w[i][:, off])
            assert rel(back(g[i][:, p]), back(w[i][:, p]))[1] < (1e-3 if weight == "f16" else 1e-5)


@pytest.mark.parametrize("weight", ["f16", "q8_0_a32", "f32"])
@pytest.mark.parametrize("lanes,cap,few,short", [(48, 1600, 1, 1600), (48, 1600, 17, 700), (24, 600, 8, 257),
                                                 (2, 512, 2, 300)])
def test_workspace_of_the_largest_serves_the_smaller(dev, weight, lanes, cap, few, short):
    layers, fn = stack.random_weights(ONE, 3)
    st = stack.Stack(ONE, layers, fn, dev, weight)
    assert all(st.workspace_bytes(n, c) <= st.workspace_bytes(n + 1, c) for n in range(1, lanes) for c in (short, cap))
    assert st.workspace_bytes(few, short) <= st.workspace_bytes(lanes, cap)
    state = st.new_state(few, short)
    ws = torch.zeros(st.workspace_bytes(lanes, cap), dtype=torch.uint8, device=dev)
    x, kc, vc = inputs(ONE, 3, few, short, weight=weight)
    pos = np.asarray([(short - 1 - i * 37) % short for i in range(few)], np.int32)
    want = oracle.stack_decode_f32(ONE, layers, fn, x, kc, vc, pos, weight)
    x, kc, vc = inputs(ONE, 3, few, short, weight=weight)
    put = to_dev if weight == "f16" else lambda a, d: torch.from_numpy(a).to(d)
    state.k[0].copy_(put(kc[0], dev))
    state.v[0].copy_(put(vc[0], dev))
    got = to_host(st.decode(to_dev(x, dev), state, pos, workspace=ws))
    torch.cuda.synchronize()
    assert rel(got, want)[1] < (2e-4 if weight == "f16" else 1e-5)
