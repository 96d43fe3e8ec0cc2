"""The fp32 products at the three row-tile heights: rows, widths and k that are no multiple of the tiles, forward and backward
against the oracle (fp32 sums of at most a few thousand terms: relative L2 within 1e-5, as for every fp32 layer)."""
import ctypes
import importlib

import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests.synth import C
from tests.test_gpu_backward import _check_grads, _setup

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")

# tiles of 128 and of 64 rows with 16-byte loads: ragged row tiles, last column tiles, partial k steps
ROWS_128 = dict(T=1333, d=228, H=228, E=3, K=3, Es=1)
ROWS_64 = dict(T=1955, d=100, H=132, E=3, K=3, Es=1)
CASES = [
    dict(T=1300, d=1028, H=68, E=3, K=3, Es=1),    # tiles of 32 rows, and of 128 x 128 in the weight gradients
    dict(T=1301, d=1027, H=67, E=3, K=3),          # the same without 16-byte loads
    dict(T=300, d=260, H=132, E=2, K=2),           # tiles of 32 rows, whole and partial k steps
    dict(T=77, d=68, H=60, E=5, K=3, Es=1),        # ragged tiles of 32 rows, one k step and a part, less than one
    dict(T=77, d=67, H=65, E=5, K=3, Es=1),        # the same without 16-byte loads
    dict(T=1, d=128, H=256, E=8, K=2),             # a row per expert
    dict(T=33, d=31, H=5, E=2, K=1),               # less than one k step
    dict(T=200, d=33, H=5, E=2, K=2),              # whole k steps of weight gradients far narrower than a tile
    dict(T=64, d=32, H=64, E=1, K=1),              # whole row tiles, half a k step and one
    dict(T=32, d=32, H=64, E=1, K=1),              # exactly one row tile, one k step of the down product
    dict(T=1333, d=228, H=235, E=3, K=3, Es=1),    # 16-byte loads in the up product alone, tiles of 128 rows
    dict(T=77, d=68, H=61, E=5, K=3, Es=1),        # and of 32
    dict(T=1333, d=235, H=228, E=3, K=3, Es=1),    # in the down product alone, tiles of 128 rows
    dict(T=77, d=67, H=60, E=5, K=3, Es=1),
    ROWS_128,
    dict(ROWS_128, d=193, H=235),                  # tiles of 128 rows without 16-byte loads
    ROWS_64,
    dict(ROWS_64, d=99, H=131),                    # of 64
]


@pytest.mark.parametrize("kw", CASES)
def test_fp32_products_match_oracle(kw):
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", kw, 77)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)
    g = G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)
    out = layer.forward(x).to_numpy()
    assert N.rel_l2(out, G.oracle_forward(cfg, inp)["out"]) < 1e-5
    dx = layer.back(g).to_numpy()
    ref = O.moe_backward(inp["x"], dout, inp["Wg"], inp["bg"], inp["W1"], inp["W3"], inp["W2"], cfg.K, cfg.renorm, cfg.Es)
    assert N.rel_l2(dx, ref["dx"]) < 1e-5
    _check_grads(layer, cfg, ref, 1e-5)
    layer.close()


@pytest.mark.parametrize("kw", [CASES[0], CASES[1], CASES[6], ROWS_128, ROWS_64, dict(T=50, d=48, H=40, E=16, K=2, zipf_bias=1.2)])
def test_fp32_training_mode_keeps_h1_h3(kw):
    """The backward pass reads the h1, h3 and probabilities that a training forward left: the same bits as computing them
    again, once; a second backward pass, whose d(a) product has overwritten them, computes them again."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", kw, 78)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)
    g = G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)

    def grads():
        return [layer.back(g).to_numpy(), layer.grad(L.W_GATE)] + [
            layer.grad(w, e) for e in range(cfg.E + cfg.Es) for w in (L.W_W1, L.W_W3, L.W_W2)]

    def same(a, b):
        return all(np.array_equal(u, v) for u, v in zip(a, b))

    out = layer.forward(x).to_numpy()
    want = grads()
    layer.set_training(True)
    assert np.array_equal(layer.forward(x).to_numpy(), out)
    assert same(grads(), want) and same(grads(), want)
    layer.forward(x)
    layer.set_training(False)      # what was kept no longer counts
    assert same(grads(), want)
    fresh = G.build_layer(cfg, inp)
    fresh.set_training(True)
    fresh.forward(x)
    with pytest.raises(RuntimeError):      # no backward pass yet: no gradients, as without training mode
        fresh.grad(L.W_GATE)
    fresh.close()
    layer.close()


@pytest.mark.parametrize("kw", [dict(T=77, d=68, H=60, E=5, K=3, Es=1), dict(T=1301, d=1027, H=67, E=3, K=3)])
def test_fp32_gather_beside_the_up_product(kw):
    """A forward pass fetches the rows of the up product from x and leaves the gathered copy beside it; the stages run one by
    one gather first.  Same bits, and the up product can run again on the copy."""
    G, cfg, inp, _, layer = _setup("c1_tiny_f32", kw, 79)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)
    out = layer.forward(x).to_numpy()
    xg, a = layer.workspace("xg", cfg.T), layer.workspace("a", cfg.T)
    assert np.array_equal(xg, inp["x"][layer.routing(cfg.T)["src_row"]])
    lib, ctx, h = layer.lib, layer.ctx, layer.handle
    xp = x.ptr if cfg.Es else None          # (shared experts read the token rows)
    ctx.check(lib.omega_moe_experts_up(h, xp, cfg.T))
    assert np.array_equal(layer.workspace("a", cfg.T), a)
    o2 = G.P.DeviceBuffer(ctx, (cfg.T, cfg.d), cfg.dtype)
    for st in (lib.omega_moe_router(h, x.ptr, cfg.T), lib.omega_moe_dispatch(h, x.ptr, cfg.T), lib.omega_moe_experts_up(h, xp, cfg.T),
               lib.omega_moe_experts_down(h, cfg.T), lib.omega_moe_combine(h, cfg.T, o2.ptr)):
        ctx.check(st)
    assert np.array_equal(o2.to_numpy(), out) and np.array_equal(layer.workspace("xg", cfg.T), xg)
    layer.close()


@pytest.mark.parametrize("d,H", [(33, 5), (68, 60)])  # groups that start on any float / on 16 bytes
def test_update_steps_every_expert(d, H):
    """w - lr * g with one rounding, every tensor of every expert (float64 rounds it twice: within 1e-7)."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(T=40, d=d, H=H, E=5, K=2, Es=1), 3)
    layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype))
    layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype))
    kinds = ((L.W_W1, "W1", (H, d)), (L.W_W3, "W3", (H, d)), (L.W_W2, "W2", (d, H)))
    grads = {(k, g): layer.grad(w, g).astype(np.float64) for w, k, _ in kinds for g in range(cfg.E + cfg.Es)}
    layer.update(0.25)
    for w, k, shape in kinds:
        for g in range(cfg.E + cfg.Es):
            assert N.rel_l2(layer._download_weight(w, g, shape), inp[k][g] - 0.25 * grads[k, g]) < 1e-7, (k, g)
    layer.close()


@pytest.mark.parametrize("training", [False, True])
def test_one_layer_at_every_tile_height(training):
    """Batches with tiles of 128 rows, then 64, 32 and 128 again on one layer's workspace: the bits of a layer that sees the batch
    alone."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", ROWS_128, 80)

    def step(lay, T):
        lay.set_training(training)
        x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"][:T], cfg.dtype)
        g = G.P.DeviceBuffer.from_numpy(G.ctx(), dout[:T], cfg.dtype)
        out = lay.forward(x).to_numpy()
        return [out, lay.back(g).to_numpy(), lay.grad(L.W_GATE)] + [
            lay.grad(w, e) for e in range(cfg.E + cfg.Es) for w in (L.W_W1, L.W_W3, L.W_W2)]

    for T in (cfg.T, 900, 77, 1, cfg.T):
        alone = G.build_layer(cfg, inp)
        assert all(np.array_equal(a, b) for a, b in zip(step(layer, T), step(alone, T))), T
        alone.close()
    layer.close()


def _chain(A, B):
    """A . B as one fp32 chain of fused multiply-adds over k, element by element."""
    s = np.zeros((A.shape[0], B.shape[1]), np.float32)
    for k in range(A.shape[1]):
        s = (A[:, k:k + 1].astype(np.float64) * B[k:k + 1].astype(np.float64) + s).astype(np.float32)
    return s


@pytest.mark.parametrize("T,d,H", [(64, 64, 3584), (64, 63, 3551), (4096, 96, 3596), (49088, 128, 3584), (49088, 128, 3620)])
def test_input_gradient_adds_two_sums(T, d, H):
    """dxg = dh1 . W1 + dh3 . W3 is the sum of two sums of H terms (tiles of 32 rows, of 64 and of 128; an odd number of k
    steps; k left over), not a chain of 2 H: against float64 the error is that of two chains on the same operands (1.2: the roundings of
    dh itself, three sums of d terms, add at most sqrt(1 + 3 d / H) = 1.05, and 4096 elements scatter by a few percent), where
    one chain has 1.41 times it."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(T=T, d=d, H=H, E=1, K=1), 81)
    layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype))
    dx = layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)).to_numpy()
    rows = np.linspace(0, T - 1, 64).astype(int)
    x, g, W1, W3, W2 = (a.astype(np.float64) for a in (inp["x"][rows], dout[rows], inp["W1"][0], inp["W3"][0], inp["W2"][0]))
    h1, h3, da = x @ W1.T, x @ W3.T, g @ W2        # one expert: combine weight 1, no gradient through the gate
    s = 1.0 / (1.0 + np.exp(-h1))
    dh1, dh3 = da * h3 * s * (1.0 + h1 * (1.0 - s)), da * h1 * s
    exact = dh1 @ W1 + dh3 @ W3
    two = _chain(dh1.astype(np.float32), inp["W1"][0]) + _chain(dh3.astype(np.float32), inp["W3"][0])
    err, two_err = N.rel_l2(dx[rows], exact), N.rel_l2(two, exact)
    assert err < 1.2 * two_err
    layer.close()


@pytest.mark.parametrize("kw", [CASES[0], ROWS_128, ROWS_64, dict(T=77, d=68, H=61, E=5, K=3, Es=1), dict(T=77, d=68, H=60, E=5, K=3)])
def test_rows_that_start_off_a_16_byte_boundary(kw):
    """The caller's x and dout one float behind an aligned address: loads element by element, the same bits."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", kw, 83)
    ctx, lib, n = layer.ctx, layer.lib, cfg.T * cfg.d
    got = []
    for skip in (0, 1):
        x, g = (G.P.DeviceBuffer.from_numpy(ctx, np.concatenate([np.zeros(skip, np.float32), a.reshape(-1)]), "f32")
                for a in (inp["x"], dout))
        out, dx = (G.P.DeviceBuffer(ctx, (cfg.T, cfg.d), "f32") for _ in range(2))
        xp, gp = (ctypes.c_void_p(b.ptr.value + 4 * skip) for b in (x, g))
        ctx.check(lib.omega_moe_forward(layer.handle, xp, cfg.T, out.ptr))
        ctx.check(lib.omega_moe_backward(layer.handle, xp, gp, cfg.T, dx.ptr))
        got.append([out.to_numpy(), dx.to_numpy(), layer.grad(L.W_GATE)] + [
            layer.grad(w, e) for e in range(cfg.E + cfg.Es) for w in (L.W_W1, L.W_W3, L.W_W2)])
    assert all(np.array_equal(a, b) for a, b in zip(*got))
    layer.close()


def test_timed_backward_passes_leave_the_gradients_of_one():
    """What a timed pass of a training step uses up is computed again in front of the next: every pass gives the same bits."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", ROWS_128, 84)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)
    g = G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)
    dx = G.P.DeviceBuffer(G.ctx(), (cfg.T, cfg.d), cfg.dtype)
    layer.set_training(True)
    layer.forward(x)
    want = [layer.back(g).to_numpy(), layer.grad(L.W_GATE), layer.grad(L.W_W1, 1), layer.grad(L.W_W2, 3)]
    layer.forward(x)
    assert layer.time_backward(x, g, cfg.T, dx, warmup=1, iters=2) > 0
    got = [dx.to_numpy(), layer.grad(L.W_GATE), layer.grad(L.W_W1, 1), layer.grad(L.W_W2, 3)]
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    layer.close()


@pytest.mark.parametrize("T,d,H,E", [(5377, 195, 483, 3), (5662, 200, 412, 3), (5087, 76, 452, 2), (2111, 724, 324, 3), (2113, 723, 323, 3)])
def test_last_round_of_tiles_in_parts(T, d, H, E):
    """An eighth of the tiles is one or two rounds of what an XCD holds (64; 128 of 64 x 64) and at most a quarter more, which goes in
    parts of 32 x 32.  Tiles of 128 rows: every product without 16-byte loads, a single row in an expert's last tile and 35 columns in a
    product's; down, d(a) and input gradient with 16-byte loads; up with them.  Of 64: up, down and input gradient."""
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(T=T, d=d, H=H, E=E, K=E), 85)
    x = G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype)
    g = G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype)
    out = layer.forward(x).to_numpy()
    ref = G.oracle_forward(cfg, inp)["out"]
    assert N.rel_l2(out, ref) < 1e-5 and N.rel_l2(out[-3:], ref[-3:]) < 1e-5
    dx = layer.back(g).to_numpy()
    ref = O.moe_backward(inp["x"], dout, inp["Wg"], inp["bg"], inp["W1"], inp["W3"], inp["W2"], cfg.K, cfg.renorm, cfg.Es)
    assert N.rel_l2(dx, ref["dx"]) < 1e-5
    _check_grads(layer, cfg, ref, 1e-5)
    layer.close()
