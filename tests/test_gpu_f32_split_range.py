"""Split fp32 products (three bf16 parts per number): what the parts cannot carry is computed again, and the shapes lie on the kernels that they are meant for."""
import importlib

import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests import test_gpu_f32_split as split
from tests.test_gpu_backward import _check_grads, _setup
from tests.test_gpu_f32_products import _chain

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")

TALL = dict(T=3300, d=516, H=700, E=2, K=2)            # tiles of 128 rows, ragged in rows, columns and k
MID = dict(T=1200, d=644, H=996, E=5, K=2)             # of 64 (up product); split dW1 and dW3
MID_DA = dict(T=1800, d=644, H=996, E=5, K=2)          # of 64, enough of them for a split d(a)
ODD = dict(T=2601, d=515, H=451, E=2, K=2, Es=1)       # 128 rows without 16-byte loads
ROWS = [(TALL, 128), (MID, 64), (MID_DA, 64), (ODD, 128)]


def _height(kw):
    layer = _setup("c1_tiny_f32", kw, 1)[4]
    rows = layer.f32_tiles(kw["T"])[0]
    layer.close()
    return rows


def test_error_of_two_k_steps():
    kw = dict(T=32766, d=515, H=33, E=1, K=1)
    assert _height(kw) == 128
    split.test_error_against_float64_is_that_of_a_chain_at_most(kw["T"], kw["d"], kw["H"])


@pytest.mark.parametrize("kw,rows", ROWS)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_infinite_and_largest_weights_at_every_height(kw, rows, value):
    assert _height(kw) == rows
    split.test_infinite_and_largest_weights(kw, value)


@pytest.mark.parametrize("kw,rows", ROWS)
def test_gradients_of_tiny_deltas_at_every_height(kw, rows):
    assert _height(kw) == rows
    split.test_gradients_of_tiny_deltas(kw)


def test_tiles_computed_again_add_two_sums():
    """Weights that make a few columns of the input gradient smaller than what three bf16 parts carry: the columns beside them, computed again, are
    still the sum of two sums (test_input_gradient_adds_two_sums has the bound), and the few are as close."""
    T, d, H = 8192, 1024, 3584
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(T=T, d=d, H=H, E=1, K=1), 94)
    layer.close()
    few = np.arange(5, d, 64)
    for w in ("W1", "W3"):
        inp[w][0][:, few] *= np.float32(2.0 ** -100)
    layer = G.build_layer(cfg, inp)
    assert layer.f32_tiles(T)[0] == 128
    layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype))
    dx = layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)).to_numpy()
    rows = np.linspace(0, T - 1, 64).astype(int)
    x, g, W1, W3, W2 = (a.astype(np.float64) for a in (inp["x"][rows], dout[rows], inp["W1"][0], inp["W3"][0], inp["W2"][0]))
    h1, h3, da = x @ W1.T, x @ W3.T, g @ W2
    s = 1.0 / (1.0 + np.exp(-h1))
    dh1, dh3 = da * h3 * s * (1.0 + h1 * (1.0 - s)), da * h1 * s
    exact = dh1 @ W1 + dh3 @ W3
    two = _chain(dh1.astype(np.float32), inp["W1"][0]) + _chain(dh3.astype(np.float32), inp["W3"][0])
    dx = dx[rows].astype(np.float64)
    for cols in (few, np.setdiff1d(np.arange(d), few)):
        assert N.rel_l2(dx[:, cols], exact[:, cols]) < 1.2 * N.rel_l2(two[:, cols].astype(np.float64), exact[:, cols])
    layer.close()


WIDE_TALL = dict(T=1500, d=1284, H=900, E=5, K=2, Es=1)   # split weight gradients; row tiles of 128 ...
WIDE_MID = dict(T=900, d=1284, H=1028, E=5, K=2, Es=1)    # ... and of 64

# powers of two on x (the gate's weights and W1 take the opposite), W3, W2 and dout that leave the results what they are but for a power of two: a
# factor of 2^-120 meets one of 2^120 in (a) up, (b) d(a), (c) d(a) and, with dh, the input gradient, (d) down and input gradient, (e) dW2
SCALES = dict(up=(-120, 120, 0, 0), da=(0, 0, 120, -120), dxg=(-120, 120, 0, -120), down=(0, -120, 120, 0), wg2=(0, 120, 0, -120))


@pytest.mark.parametrize("kw,rows", [(WIDE_TALL, 128), (WIDE_MID, 64), (dict(WIDE_TALL, d=1285, H=899), 128)])
def test_tiny_factors_with_large_ones(kw, rows):
    """Scaling by powers of two is exact in fp32 as long as nothing under- or overflows: the same results but for that power, to the error of fp32
    sums in another order (K = 1285: 2e-6; factors of 2^-120 in three bf16 parts have 2e-5 and more)."""
    G, cfg, inp, dout, _ = _setup("c1_tiny_f32", kw, 96)

    def step(ex, e3, e2, eo):
        two = [np.float32(2.0 ** e) for e in (ex, e3, e2, eo, -ex)]
        p = dict(inp, x=inp["x"] * two[0], Wg=inp["Wg"] * two[4], W1=[w * two[4] for w in inp["W1"]], W3=[w * two[1] for w in inp["W3"]],
                 W2=[w * two[2] for w in inp["W2"]])
        layer = G.build_layer(cfg, p)
        assert layer.f32_tiles(cfg.T) == (rows, 128, 128)
        r = [layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), p["x"], cfg.dtype)).to_numpy(),
             layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout * two[3], cfg.dtype)).to_numpy()]
        r += [layer.grad(w, g) for g in (0, cfg.E) for w in (L.W_W1, L.W_W3, L.W_W2)]
        layer.close()
        return r

    want = step(0, 0, 0, 0)
    for name, (ex, e3, e2, eo) in SCALES.items():
        a, h = ex + e3, eo + e2                                 # of a, and of d(a)
        power = [a + e2, h + e3] + 2 * [h + e3 + 2 * ex, h + ex, eo + a]
        for got, ref, e in zip(step(ex, e3, e2, eo), want, power):
            if -100 < e < 126:
                assert N.rel_l2(got.astype(np.float64) * 2.0 ** -e, ref) < 2e-6, (name, e)


def test_weight_gradient_of_a_single_row_is_rounded_once():
    """An expert with one row in a batch whose weight gradients are split: every element is one product, rounded once."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(T=512, d=1664, H=1664, E=2, K=1), 97)
    layer.close()
    t = 7
    inp["x"][:, 0], inp["x"][t, 0] = -1.0, 1.0
    inp["Wg"][:] = 0.0
    inp["Wg"][1, 0] = 1.0
    layer = G.build_layer(cfg, inp)
    assert layer.f32_tiles(cfg.T)[1:] == (128, 128)
    layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype))
    assert layer.routing()["counts"].tolist() == [511, 1]
    a = layer.workspace("a", cfg.T)[-1]
    layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype))
    assert np.array_equal(layer.grad(L.W_W2, 1), dout[t][:, None] * a[None, :])
    layer.close()


@pytest.mark.parametrize("kw,rows", ROWS)
@pytest.mark.parametrize("place,zeros", [(0, False), (0, True), (41, False), (41, True), (-1, True)])
def test_tiny_factors_among_zeros(kw, rows, place, zeros):
    """A column of x times 2^-120 that meets one of W1 and W3 times 2^120, in the first k step, a later one and the last, partial one, in a batch that has
    zeros from its first step on and in one that has none: the same results (as test_tiny_factors_with_large_ones)."""
    G, cfg, inp, dout, _ = _setup("c1_tiny_f32", kw, 98)
    if zeros:
        inp["x"][::8], dout[3::8] = 0.0, 0.0
    inp["Wg"][:, place] = 0.0

    def step(e):
        two, inv = np.float32(2.0 ** e), np.float32(2.0 ** -e)
        p = dict(inp, x=inp["x"].copy(), W1=[w.copy() for w in inp["W1"]], W3=[w.copy() for w in inp["W3"]])
        p["x"][:, place] *= two
        for w in p["W1"] + p["W3"]:
            w[:, place] *= inv
        layer = G.build_layer(cfg, p)
        assert layer.f32_tiles(cfg.T)[0] == rows
        out = layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), p["x"], cfg.dtype)).to_numpy()
        dx = layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)).to_numpy().astype(np.float64)
        dx[:, place] *= 2.0 ** e
        r = [out, dx, layer.grad(L.W_W2, 0), np.delete(layer.grad(L.W_W1, 1), place, 1)]
        layer.close()
        return r

    for got, ref in zip(step(-120), step(0)):
        assert N.rel_l2(got, ref) < 2e-6


@pytest.mark.parametrize("d,H,Es", [(900, 1300, 1), (899, 1301, 1), (900, 1300, 0)])
def test_split_weight_gradients_match_oracle(d, H, Es):
    """Every expert's gradients: all rows, all but ten of them, ten and none; a shared expert, whose rows are the tokens."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(T=300, d=d, H=H, E=4, K=2, Es=Es), 99)
    layer.close()
    inp["Wg"][:], inp["x"][:, 0], inp["x"][:, 1] = 0.0, 1.0, 0.0
    inp["Wg"][:, 0], inp["Wg"][2, 1] = (3.0, 2.0, 0.0, -9.0), 2.5
    inp["x"][17:187:17, 1] = 1.0
    layer = G.build_layer(cfg, inp)
    assert layer.f32_tiles(cfg.T)[1:] == (128, 128)
    layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype))
    assert layer.routing()["counts"].tolist() == [300, 290, 10, 0]
    dx = layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)).to_numpy()
    ref = O.moe_backward(inp["x"], dout, inp["Wg"], inp["bg"], inp["W1"], inp["W3"], inp["W2"], cfg.K, cfg.renorm, cfg.Es)
    assert N.rel_l2(dx, ref["dx"]) < 1e-5
    _check_grads(layer, cfg, ref, 1e-5)
    layer.close()
