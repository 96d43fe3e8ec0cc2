"""fp32 products on the bf16 matrix cores: error against float64, and sums that three bf16 parts cannot carry."""
import importlib

import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests.test_gpu_backward import _setup
from tests.test_gpu_f32_products import _chain

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")

TALL = dict(T=2600, d=516, H=452, E=2, K=2)            # tiles of 128 rows, ragged in rows, columns and k
MID = dict(T=1450, d=644, H=996, E=5, K=2)             # of 64 (up product and d(a))
ODD = dict(T=2601, d=515, H=451, E=2, K=2, Es=1)       # without 16-byte loads


@pytest.mark.parametrize("T,d,H", [(8192, 128, 3584), (8192, 1024, 1100), (8190, 131, 33)])
def test_error_against_float64_is_that_of_a_chain_at_most(T, d, H):
    """y of the down product, on the layer's own `a`: no further from float64 than a chain of fp32 fused multiply-adds (1.05: 64 rows
    scatter by a few percent)."""
    G, cfg, inp, _, layer = _setup("c1_tiny_f32", dict(T=T, d=d, H=H, E=1, K=1), 91)
    layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype))
    rows = np.linspace(0, T - 1, 64).astype(int)
    a, y = layer.workspace("a", T)[rows], layer.workspace("y", T)[rows]
    W2 = inp["W2"][0]
    exact = a.astype(np.float64) @ W2.astype(np.float64).T
    assert N.rel_l2(y, exact) < 1.05 * N.rel_l2(_chain(a, np.ascontiguousarray(W2.T)), exact)
    layer.close()


@pytest.mark.parametrize("kw", [TALL, MID, ODD])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_infinite_and_largest_weights(kw, value):
    """One element of W1: what the oracle makes infinite or no number is that here, and nothing else (3.4e38 rounds to an infinite bf16)."""
    G, cfg, inp, _, _ = _setup("c1_tiny_f32", kw, 92)
    inp["W1"][0][7, 3] = value
    layer = G.build_layer(cfg, inp)
    out = layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)).to_numpy()
    with np.errstate(all="ignore"):
        ref = G.oracle_forward(cfg, inp)["out"]
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(out), f(ref))
    out, ref = out.astype(np.float64), ref.astype(np.float64)
    finite, large = np.isfinite(ref).all(axis=1), np.abs(ref).max(axis=1) > 1e6
    for rows in (finite & large, finite & ~large):      # (the large weight's rows outweigh the others by far)
        assert not rows.any() or N.rel_l2(out[rows], ref[rows]) < 1e-5
    layer.close()


@pytest.mark.parametrize("kw", [TALL, MID, ODD])
def test_gradients_of_tiny_deltas(kw):
    """The gradients are linear in dout: with dout times 2^-100, whose products' factors lie below what three bf16 parts hold, they are
    those of dout times 2^-100 (no fp32 denormals there: gradients of 1e-4 and more)."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", kw, 93)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)
    s = np.float32(2.0 ** -100)
    got = []
    for f in (np.float32(1), s):
        layer.forward(x)
        dx = layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout * f, cfg.dtype)).to_numpy()
        got.append([dx] + [layer.grad(w, 0) for w in (L.W_W1, L.W_W3, L.W_W2)])
    for a, b in zip(*got):
        assert N.rel_l2(b.astype(np.float64) / float(s), a) < 1e-5
    layer.close()
