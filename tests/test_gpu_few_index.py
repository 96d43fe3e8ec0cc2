"""The dispatch index that the up launch of a few-token batch makes is the one of a dispatch stage of its own, at the edges of what it takes
(1024 pairs, 64 tokens, 256 experts, 64 choices a token) and one beyond."""
import numpy as np
import pytest

from oracle import oracle_np as N
from tests.test_gpu_few_tokens import _layer

pytestmark = pytest.mark.gpu

SHAPES = [
    dict(T=1, E=1, K=1, Es=0), dict(T=64, E=1, K=1, Es=1), dict(T=1, E=256, K=64, Es=0), dict(T=16, E=64, K=64, Es=0),
    dict(T=17, E=70, K=64, Es=1), dict(T=64, E=200, K=16, Es=0), dict(T=64, E=256, K=16, Es=64), dict(T=63, E=255, K=16, Es=2),
    dict(T=33, E=33, K=31, Es=0), dict(T=64, E=130, K=8, Es=1, zipf_bias=1.2),
]


@pytest.mark.parametrize("kw", SHAPES, ids=lambda k: "-".join(str(v) for v in k.values()))
def test_index_of_the_up_launch(kw):
    G, cfg, inp, layer, x = _layer(dict(kw, d=256, H=256), 15, 1)
    out = layer.forward(x).to_numpy()
    got, xg = layer.routing(), layer.workspace("xg", cfg.T)
    layer.fill_workspace("a", 0xFF)
    layer.fill_workspace("y", 0xFF)
    o = G.P.DeviceBuffer(G.ctx(), (cfg.T, cfg.d), cfg.dtype)
    for s in ("router", "dispatch", "experts"):
        layer.stage(s, x)
    layer.stage("combine", out=o)
    want = layer.routing()
    assert all(np.array_equal(got[k], want[k]) for k in want)
    assert np.array_equal(o.to_numpy(), out) and np.array_equal(layer.workspace("xg", cfg.T), xg)
    ref = G.oracle_forward(cfg, inp)
    G.assert_routing_bit_exact(got, ref)
    assert N.rel_l2(out, ref["out"]) <= 1e-2
    x.free()
    o.free()
    layer.close()


@pytest.mark.parametrize("kw", [dict(T=4, E=161, K=32, H=1664, Es=1), dict(T=15, E=163, K=20, H=1792, Es=0)])
def test_both_sides_of_the_work_limit(kw):
    """1.7 and 5.5 million pairs x workgroups: an index by the up launch, and by a launch of its own (makes_index_in_up)."""
    G, cfg, inp, layer, x = _layer(dict(kw, d=256), 16, 1)
    out = layer.forward(x).to_numpy()
    got = layer.routing()
    ref = G.oracle_forward(cfg, inp)
    G.assert_routing_bit_exact(got, ref)
    assert N.rel_l2(out, ref["out"]) <= 1e-2
    x.free()
    layer.close()
