"""Block form, forward and backward, at the edges of the row kernels of the norm (two rows per workgroup, one, or rows in
chunks; widths that leave pieces of a thread unused) and of the gate-gradient kernel (experts behind a unit of 32, columns
behind a block of 256, token slices of odd length).  Row statistics bit for bit; gradients within the fp32 (1e-5) and bf16
(1e-2) relative L2 of every layer test."""
import importlib

import numpy as np
import pytest

from oracle import oracle_np as N
from tests.test_gpu_block import test_block_backward_matches_oracle as block_backward
from tests.test_gpu_block import test_block_forward_matches_oracle as block_forward

pytestmark = pytest.mark.gpu
L = importlib.import_module("omega-ai_amd._lib")

F32 = dict(E=3, K=2, H=32, Es=0, dtype="f32", renorm=True)
CASES = [
    ("c1_tiny_f32", dict(F32, T=1, d=8)),
    ("c1_tiny_f32", dict(F32, T=35, d=1000)),                  # 250 pieces for 256 threads
    ("c1_tiny_f32", dict(F32, T=21, d=2056, E=33, K=3)),       # one expert behind the unit of 32
    ("c1_tiny_f32", dict(F32, T=9, d=4104)),                   # one row per workgroup
    ("c1_tiny_f32", dict(F32, T=9, d=8200)),                   # rows in chunks
    ("c2_mixtral", dict(T=33, d=4096, H=256, E=2, K=1)),
    ("c2_mixtral", dict(T=17, d=8192, H=256, E=1, K=1)),
    ("c5_skewed", dict(T=131, d=768, H=256, E=70, K=5)),
]


@pytest.mark.parametrize("name,kw", CASES)
def test_block_backward(name, kw):
    block_backward(name, kw, True)


@pytest.mark.parametrize("name,kw", CASES)
def test_block_forward(name, kw):
    block_forward(name, kw)


@pytest.mark.parametrize("T,d", [(4096, 4096), (1500, 8192)])
def test_gate_gradient_of_wide_layers_keeps_its_slices(T, d):
    """dWg = dlogits^T x of 256 experts and wide rows against float64, on the dlogits of the pass: no more rounding error than 32
    partial sums over the tokens, each one chain, added in order (1.1: the 16384 elements that are compared scatter by a few
    percent; a chain twice as long has 1.25 times the error)."""
    from tests.test_gpu_backward import _setup
    G, cfg, inp, dout, layer = _setup("c1_tiny_f32", dict(T=T, d=d, E=256, K=2, H=8, renorm=False), 82)
    layer.set_gate(inp["Wg"] / np.float32(d ** 0.5 / 8), None)     # a spread of 1, and no renormalisation: every token counts
    layer.forward(G.P.DeviceBuffer.from_numpy(G.ctx(), inp["x"], cfg.dtype))
    layer.back(G.P.DeviceBuffer.from_numpy(G.ctx(), dout, cfg.dtype))
    dl, cols = layer.workspace("dlogits", T), slice(100, 164)
    x, got = inp["x"][:, cols], layer.grad(L.W_GATE)[:, cols]
    exact = dl.astype(np.float64).T @ x.astype(np.float64)
    total = np.zeros_like(got)
    step = -(-T // 32)
    for t0 in range(0, T, step):
        s = np.zeros_like(got)
        for t in range(t0, min(T, t0 + step)):
            s = (dl[t][:, None].astype(np.float64) * x[t][None, :] + s).astype(np.float32)
        total += s
    err, want = N.rel_l2(got, exact), N.rel_l2(total, exact)
    assert err < 1.1 * want
    layer.close()
