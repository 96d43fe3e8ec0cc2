"""The k slices of a down product that the combine kernel adds: the bits of the kernel that adds them into y, every tile sliced, the
last tiles only, none, with shared experts, and behind an output that only the element-wise combine can write."""
import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests.synth import C, scaled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [
    dict(T=70, d=512, H=1024, E=4, K=2, Es=0),      # 4 slices of every tile
    dict(T=90, d=768, H=4096, E=3, K=3, Es=2),      # 8 slices, shared experts
    dict(T=300, d=1024, H=640, E=7, K=7, Es=1),     # 2 slices, two row tiles per expert
    dict(T=200, d=1024, H=2048, E=8, K=6, Es=2),    # 6 slices, eight rows in two groups
    dict(T=130, d=512, H=1024, E=5, K=4, Es=1),     # five rows in groups of three
    dict(T=300, d=2048, H=1408, E=64, K=6, Es=2),   # room for slices, and none made: too many tiles
    dict(T=4400, d=4096, H=4096, E=1, K=1, Es=0),   # the last tiles only: 18 x 16 tiles, 32 of them in 2 slices
    dict(T=1100, d=256, H=256, E=4, K=1, Es=0),     # items of 128 columns, no slices
], ids=lambda k: "-".join(str(v) for v in k.values()))
def test_combine_adds_the_k_slices(kw):
    """The sums the combine kernel forms from y and the slices are those of the kernel that adds them into y: the same bits."""
    from tests import gpu_util as G
    cfg = scaled(C.CONFIGS["c4_finegrained"], **kw)
    layer = G.P.MoELayer(cfg.d, cfg.H, cfg.E, cfg.K, renorm=cfg.renorm, nShared=cfg.Es, bias=False, ctx=G.ctx(), dtype="bf16")
    layer.init_synthetic(13, C, cfg)
    x = G.P.DeviceBuffer(G.ctx(), (cfg.T, cfg.d), "bf16")
    x.fill_normal(13, C.STREAM_X, 1.0)
    out = layer.forward(x).to_numpy()
    y = layer.workspace("y", cfg.T)             # adds the slices into y
    o = G.P.DeviceBuffer(G.ctx(), (cfg.T * cfg.d + 8,), "bf16")
    layer.ctx.check(layer.lib.omega_moe_combine(layer.handle, cfg.T, o.ptr))
    assert np.array_equal(o.to_numpy()[:cfg.T * cfg.d].reshape(cfg.T, cfg.d), out)
    assert np.array_equal(layer.workspace("y", cfg.T), y)
    # an output off the 16-byte boundary: the element-wise combine needs y whole
    layer.ctx.check(layer.lib.omega_moe_forward(layer.handle, x.ptr, cfg.T, o.ptr.value + 2))
    assert np.array_equal(o.to_numpy()[1:cfg.T * cfg.d + 1].reshape(cfg.T, cfg.d), out)
    # rows by the definition, from the layer's own y
    r = layer.routing()
    t = np.arange(0, cfg.T, max(1, cfg.T // 16))
    ref = np.zeros((len(t), cfg.d))
    for j in range(cfg.K):
        ref += r["w"][t, j, None].astype(np.float64) * y[r["dst"].reshape(cfg.T, cfg.K)[t, j]]
    for s in range(cfg.Es):
        ref += y[cfg.T * cfg.K + s * cfg.T + t]
    assert N.rel_l2(out[t], ref) <= 4e-3        # one rounding to bf16: at most 2^-9 of an element
    for b in (o, x):
        b.free()
    layer.close()


def test_a_batch_without_slices_behind_one_with_them():
    """4400 tokens leave a last round of 32 tiles, in 2 slices each; 4096 are one whole round: room for slices, and none made, but y_slabs
    and the table of the batch before are still there.  Then the first again."""
    from tests import gpu_util as G
    cfg = scaled(C.CONFIGS["c4_finegrained"], T=4400, d=4096, H=4096, E=1, K=1, Es=0)

    def build():
        layer = G.P.MoELayer(cfg.d, cfg.H, cfg.E, cfg.K, renorm=cfg.renorm, nShared=cfg.Es, bias=False, ctx=G.ctx(), dtype="bf16")
        layer.init_synthetic(17, C, cfg)
        return layer

    layer = build()
    x = G.P.DeviceBuffer(G.ctx(), (cfg.T, cfg.d), "bf16")
    x.fill_normal(17, C.STREAM_X, 1.0)
    bits = x.to_numpy()
    for T in (4400, 4096, 4400):
        xt = G.P.DeviceBuffer.from_numpy(G.ctx(), bits[:T], "bf16")
        out = layer.forward(xt).to_numpy()
        y = layer.workspace("y", T)                     # one expert, combine weight 1: the output is y
        assert np.array_equal(out, O.round_bf16(y)), T
        alone = build()
        assert np.array_equal(alone.forward(xt).to_numpy(), out), T
        alone.close()
        xt.free()
    x.free()
    layer.close()
