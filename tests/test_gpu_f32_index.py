"""The dispatch index that the up launch of a small fp32 batch makes is the one of a dispatch stage of its own, at the edges of what it takes (1024
pairs, 16 experts, several row tiles per expert) and one beyond."""
import numpy as np
import pytest

from oracle import oracle_np as N
from tests.test_gpu_backward import _check_grads, _setup
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [
    dict(T=1, E=1, K=1), dict(T=127, E=1, K=1, Es=2), dict(T=512, E=16, K=2, Es=1), dict(T=513, E=16, K=2), dict(T=128, E=16, K=8),
    dict(T=64, E=16, K=16, Es=1), dict(T=65, E=16, K=16), dict(T=1024, E=9, K=1), dict(T=100, E=17, K=4), dict(T=200, E=16, K=2, zipf_bias=1.2),
    dict(T=31, E=3, K=3), dict(T=33, E=13, K=7, Es=2),
]


@pytest.mark.parametrize("d,H", [(64, 96), (67, 33)])
@pytest.mark.parametrize("kw", SHAPES, ids=lambda k: "-".join(str(v) for v in k.values()))
def test_index_of_the_up_launch(kw, d, H):
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(kw, d=d, H=H), 95)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)
    out = layer.forward(x).to_numpy()
    got, xg, y = layer.routing(), layer.workspace("xg", cfg.T), layer.workspace("y", cfg.T)
    dx = layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)).to_numpy()
    ref, bw = G.oracle_forward(cfg, inp), O.moe_backward(inp["x"], dout, inp["Wg"], inp["bg"], inp["W1"], inp["W3"], inp["W2"], cfg.K, cfg.renorm, cfg.Es)
    G.assert_routing_bit_exact(got, ref)
    assert N.rel_l2(out, ref["out"]) < 1e-5 and N.rel_l2(dx, bw["dx"]) < 1e-5
    _check_grads(layer, cfg, bw, 1e-5)
    assert np.array_equal(xg, inp["x"][got["src_row"]])
    layer.fill_workspace("a", 0xFF)
    layer.fill_workspace("y", 0xFF)
    o = G.P.DeviceBuffer(G.ctx(), (cfg.T, cfg.d), cfg.dtype)
    for s in ("router", "dispatch", "experts"):
        layer.stage(s, x)
    layer.stage("combine", out=o)
    want = layer.routing()
    assert all(np.array_equal(got[k], want[k]) for k in want)
    assert np.array_equal(o.to_numpy(), out) and np.array_equal(layer.workspace("xg", cfg.T), xg) and np.array_equal(layer.workspace("y", cfg.T), y)
    layer.close()
