"""Weight gradients on the four-wave kernel (24 tiles per workgroup and more): an H of 128 mod 256, experts without rows, with
less than one item's k steps and with several row tiles.  The products' operands are bf16 rows of the workspace, so float64
gives them exactly; the sums are fp32 over at most a few hundred rows (relative L2 far below 1e-5)."""
import importlib

import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests.synth import C, scaled

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")


@pytest.mark.parametrize("kw", [
    dict(T=600, d=2048, H=896, E=192, K=4, zipf_bias=1.2),   # both products
    dict(T=70, d=1024, H=896, E=224, K=2, zipf_bias=0.0),    # dW1 and dW3 only: dW2 has 14 tiles per workgroup
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
    a, xg, dh = (layer.workspace(n, T).astype(np.float64) for n in ("a", "xg", "dh"))
    dy = np.empty((T * K, d))
    dy[r["dst"]] = O.round_bf16(r["w"].reshape(-1)[:, None] * np.repeat(g.to_numpy(), K, axis=0))
    off, n = r["offsets"], np.diff(r["offsets"])
    for e in sorted({int(n.argmin()), int(n.argmax()), int(np.argsort(n)[E // 2]), E - 1}):
        s = slice(off[e], off[e + 1])
        for got, want in ((layer.grad(L.W_W2, e), dy[s].T @ a[s]), (layer.grad(L.W_W1, e), dh[s, :H].T @ xg[s]),
                          (layer.grad(L.W_W3, e), dh[s, H:].T @ xg[s])):
            if n[e] == 0:
                assert not got.any(), e
            else:
                assert N.rel_l2(got, want) < 1e-5, (e, int(n[e]))
    layer.close()
    x.free()
    g.free()
