"""Batches of a few tokens on bf16 layers (at most 64: the products stream the weights into registers, waves sharing k) and the
k slices that the combine kernel adds, at the sizes where they can go wrong: token counts at the edges of a unit of 16 rows, of
the kernel's variants and of the path itself, k steps that the waves cannot share evenly, widths with one column block more or
less, experts without rows, shared experts.  Every 32-row block of `a` and `y` against float64 dot products of the layer's own
operands (gpu_util), outputs and gradients within the 1e-2 relative L2 of every bf16 test."""
import importlib

import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests.synth import C, make_inputs, scaled

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")

FINE = dict(d=512, H=640, E=16, K=4, Es=2)
SHAPES = [dict(FINE, T=t) for t in (1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65)] + [
    dict(T=5, d=256, H=256, E=4, K=1, Es=0),       # 8 k steps, as many as the down product's waves
    dict(T=64, d=1280, H=384, E=3, K=3, Es=0),     # every expert has every token; 40 and 12 k steps
    dict(T=40, d=768, H=1408, E=128, K=8, Es=1),   # most experts get a row or two
    dict(T=24, d=2048, H=4096, E=9, K=2, Es=0),    # four column blocks per workgroup
    dict(T=1, d=4096, H=512, E=2, K=2, Es=2),
]


def _layer(kw, seed, mode=0):
    from tests import gpu_util as G
    cfg = scaled(C.CONFIGS["c4_finegrained"], **kw)
    inp = make_inputs(cfg, seed)
    layer = G.build_layer(cfg, inp)
    layer.set_gather_mode(mode)
    return G, cfg, inp, layer, G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("kw", SHAPES, ids=lambda k: "-".join(str(v) for v in k.values()))
def test_few_tokens(kw, mode):
    G, cfg, inp, layer, x = _layer(kw, 11, mode)
    layer.forward(x)
    layer.fill_workspace("a", 0xFF)
    layer.fill_workspace("y", 0xFF)
    out = layer.forward(x).to_numpy()
    r, ref = layer.routing(), G.oracle_forward(cfg, inp)
    G.assert_routing_bit_exact(r, ref)
    assert np.array_equal(layer.workspace("xg", cfg.T), inp["x"][r["src_row"]])
    assert G.check_products_every_block(layer, cfg, cfg.T, r, inp["x"]) > 0
    assert N.rel_l2(out, ref["out"]) <= 1e-2
    # the stages by themselves follow the tables a forward pass leaves, and those of a dispatch of their own
    y = layer.workspace("y", cfg.T)
    layer.fill_workspace("a", 0xFF)
    layer.fill_workspace("y", 0xFF)
    layer.stage("experts", x)
    assert np.array_equal(layer.workspace("y", cfg.T), y)
    o = G.P.DeviceBuffer(G.ctx(), (cfg.T, cfg.d), cfg.dtype)
    for s in ("router", "dispatch", "experts"):
        layer.stage(s, x)
    layer.stage("combine", out=o)
    assert N.rel_l2(o.to_numpy(), ref["out"]) <= 1e-2
    assert np.array_equal(layer.forward(x).to_numpy(), out)
    for b in (o, x):
        b.free()
    layer.close()


@pytest.mark.parametrize("T", [1, 33, 64])
def test_backward_behind_a_forward_of_few_tokens(T):
    """The tile kernels' queues are made when the backward pass asks for them."""
    G, cfg, inp, layer, x = _layer(dict(FINE, T=T), 12)
    dout = O.round_bf16(O.fill_normal(T * cfg.d, 12, 900, 1.0).reshape(T, cfg.d))
    layer.forward(x)
    dx = layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)).to_numpy()
    bw = O.moe_backward(inp["x"], dout, inp["Wg"], inp["bg"], inp["W1"], inp["W3"], inp["W2"], cfg.K, cfg.renorm, cfg.Es, bf16=True)
    assert N.rel_l2(dx, bw["dx"]) <= 1e-2
    for g in range(cfg.E + cfg.Es):
        for which, name in ((L.W_W1, "dW1"), (L.W_W3, "dW3"), (L.W_W2, "dW2")):
            assert N.rel_l2(layer.grad(which, g), bw[name][g]) <= 1e-2, (g, name)
    x.free()
    layer.close()


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("kw", [dict(FINE, T=1), dict(FINE, T=17), dict(FINE, T=64), dict(T=33, d=256, H=384, E=5, K=2, Es=0)],
                         ids=lambda k: "-".join(str(v) for v in k.values()))
def test_stages_of_a_few_tokens_are_those_of_a_forward_pass(kw, mode):
    """Called one by one they run on the same kernels, from the rows the dispatch stage has copied or left: the same bits."""
    G, cfg, inp, layer, x = _layer(kw, 13, mode)
    out = layer.forward(x).to_numpy()
    y, a = layer.workspace("y", cfg.T), layer.workspace("a", cfg.T)
    for w in ("a", "y"):
        layer.fill_workspace(w, 0xFF)
    o = G.P.DeviceBuffer(G.ctx(), (cfg.T, cfg.d), cfg.dtype)
    for s in ("router", "dispatch", "experts"):
        layer.stage(s, x)
    layer.stage("combine", out=o)
    assert np.array_equal(o.to_numpy(), out)
    assert np.array_equal(layer.workspace("a", cfg.T), a) and np.array_equal(layer.workspace("y", cfg.T), y)
    assert np.array_equal(layer.workspace("xg", cfg.T), inp["x"][layer.routing()["src_row"]])
    # ... and still are behind a backward pass, which has the tile kernels' queues made
    assert np.array_equal(layer.forward(x).to_numpy(), out)
    layer.back(x)
    layer.stage("experts", x)
    assert np.array_equal(layer.workspace("y", cfg.T), y)
    for b in (o, x):
        b.free()
    layer.close()
