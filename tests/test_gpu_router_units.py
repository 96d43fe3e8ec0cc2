"""Exact router of bf16 layers with more than 16 experts: logits and probabilities bit for bit at the edges of its token tiles
(16 up to one per compute unit, then 32), of its expert units of 16 and at every padded expert count; a gate set anew is
the gate that is used; rows that start off a 16-byte boundary."""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest

from oracle import oracle as O
from tests.synth import C

pytestmark = pytest.mark.gpu

CASES = [(1, 256, 17, 1), (15, 512, 32, 4), (33, 256, 33, 5), (17, 768, 64, 6), (49, 2048, 64, 6), (70, 256, 100, 8),
         (31, 512, 128, 8), (40, 256, 129, 3), (65, 256, 256, 8),
         (4097, 256, 32, 2), (4111, 256, 64, 6), (4100, 256, 128, 8), (4129, 256, 200, 4)]


@pytest.mark.parametrize("T,d,E,K", CASES)
def test_exact_logits_bit_for_bit(T, d, E, K):
    from tests import gpu_util as G
    layer = G.P.MoELayer(d, 256, E, K, bias=True, ctx=G.ctx(), dtype="bf16")
    bg = O.fill_normal(E, 5, 9, 0.5)
    x = O.round_bf16(O.fill_normal(T * d + 1, 5, C.STREAM_X, 1.0))
    buf = G.P.DeviceBuffer.from_numpy(G.ctx(), x, "bf16")
    for seed, skip in ((5, 0), (6, 1)):  # the second time with another gate and from the second element on
        Wg = O.round_bf16(O.fill_normal(E * d, seed, C.STREAM_WG, 0.05).reshape(E, d))
        layer.set_gate(Wg, bg)
        xs = x[skip:skip + T * d].reshape(T, d)
        logits, probs = layer.router_probs(SimpleNamespace(ptr=ctypes.c_void_p(buf.ptr.value + 2 * skip)), T)
        want = O.gate(xs, Wg, bg)
        assert np.array_equal(logits.view(np.uint32), want.view(np.uint32))
        assert np.array_equal(probs.view(np.uint32), O.softmax(want).view(np.uint32))
    buf.free()
    layer.close()
