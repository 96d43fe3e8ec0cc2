"""Weight gradients of many tiles on either kernel - four waves from 1024 rows per expert, 2 tiles per workgroup and expert and 32 in
all on, else eight: an H of 128 mod 256, experts without rows, with less than one item's k steps and with several row tiles.
The products' operands are bf16 rows of the workspace, so float64 gives them exactly; the sums are fp32 over at most a few thousand
rows, added in up to 1000 products of 32 terms (relative L2 below 1e-5)."""
import importlib

import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests.synth import C, scaled

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")


@pytest.mark.parametrize("kw", [
    dict(T=600, d=2048, H=896, E=192, K=4, zipf_bias=1.2),   # few rows per expert: eight waves
    dict(T=70, d=1024, H=896, E=224, K=2, zipf_bias=0.0),
    dict(T=8200, d=4096, H=8064, E=16, K=2, zipf_bias=1.2),  # both products on four waves (512 and 1008 tiles per expert)
])
def test_weight_gradients_of_many_tiles(kw):
    from tests import gpu_util as G
    P = G.P
    cfg = scaled(C.CONFIGS["c5_skewed"], **kw)
    T, d, H, E, K = cfg.T, cfg.d, cfg.H, cfg.E, cfg.K
    layer = P.MoELayer(d, H, E, K, renorm=cfg.renorm, nShared=0, bias=cfg.has_gate_bias, ctx=G.ctx(), dtype="bf16",
                       router_mode="exact", T_max=T)
    layer.init_synthetic(5, C, cfg)
    x, g = (P.DeviceBuffer(G.ctx(), (T, d), "bf16") for _ in range(2))
    x.fill_normal(5, C.STREAM_X, C.tensor_std(cfg, "x"))
    g.fill_normal(5, 900, 1.0)
    layer.forward(x)
    layer.back(g)
    r = layer.routing()
    a, xg, dh = (layer.workspace(n, T) for n in ("a", "xg", "dh"))
    dout = g.to_numpy()
    off, n = r["offsets"], np.diff(r["offsets"])
    token, w = r["src_row"], np.empty(T * K, np.float32)
    w[r["dst"]] = r["w"].reshape(-1)
    # columns of every width: all of them, or of a wide layer the first and last 64 and 64 around the middle
    cols = lambda size: np.arange(size) if size <= 2048 else np.r_[0:64, size // 2 - 32:size // 2 + 32, size - 64:size]
    cd, cH = cols(d), cols(H)
    for e in sorted({int(n.argmin()), int(n.argmax()), int(np.argsort(n)[E // 2]), E - 1}):
        s = slice(off[e], off[e + 1])
        dy = O.round_bf16(w[s, None] * dout[token[s]][:, cd]).astype(np.float64)
        ae, xe = a[s][:, cH].astype(np.float64), xg[s][:, cd].astype(np.float64)
        d1, d3 = dh[s][:, cH].astype(np.float64), dh[s][:, H + cH].astype(np.float64)
        for got, want in ((layer.grad(L.W_W2, e)[np.ix_(cd, cH)], dy.T @ ae), (layer.grad(L.W_W1, e)[np.ix_(cH, cd)], d1.T @ xe),
                          (layer.grad(L.W_W3, e)[np.ix_(cH, cd)], d3.T @ xe)):
            if n[e] == 0:
                assert not got.any(), e
            else:
                assert N.rel_l2(got, want) < 1e-5, (e, int(n[e]))
    layer.close()
    x.free()
    g.free()
