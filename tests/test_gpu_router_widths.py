"""Exact router of layers whose width is no multiple of the staged chunk (bf16, up to 16 experts: an odd multiple of 256; fp32: whole
16-byte vectors, the last chunk partly or not reached) and the combine kernel's column shares at such widths: routing and logits bit
for bit the oracle's, outputs within the relative L2 of every layer test."""
import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle_np as N
from tests.synth import C, scaled
from tests.test_gpu_router_units import test_exact_logits_bit_for_bit as logits_bit_for_bit

pytestmark = pytest.mark.gpu

SMALL = dict(H=256, K=2, Es=1)
CASES = [("c2_mixtral", dict(SMALL, T=t, d=d, E=e)) for t, d, e in (
    (1, 256, 8), (17, 256, 16), (16, 768, 3), (33, 1280, 16), (70, 3328, 7), (5, 1792, 9), (4101, 768, 4), (100, 4864, 5))]
CASES += [("c1_tiny_f32", dict(T=t, d=d, E=e, H=24, K=2, Es=1)) for t, d, e in (
    (1, 4, 2), (16, 36, 8), (17, 64, 9), (40, 100, 16), (9, 128, 8), (33, 516, 8), (5, 1020, 16), (20, 260, 40), (7, 68, 200), (3, 63, 8))]


@pytest.mark.parametrize("name,kw", CASES)
def test_widths_between_chunks(name, kw):
    from tests import gpu_util as G
    cfg = scaled(C.CONFIGS[name], **kw)
    layer, x, out, r, ref, inp = G.run_case(cfg, seed=31)
    G.assert_routing_bit_exact(r, ref)
    lg, _ = layer.router_probs(x, cfg.T)
    z = O.gate(inp["x"], inp["Wg"], inp["bg"])
    assert np.array_equal(lg.view(np.uint32), z.view(np.uint32))
    assert N.rel_l2(out, ref["out"]) <= (1e-2 if cfg.dtype == "bf16" else 1e-5)
    x.free()
    layer.close()


# the sums split by experts: 4, 8 and 16 tokens per workgroup, a last group of one expert, of fifteen, ragged token groups
@pytest.mark.parametrize("T,d,E,K", [(3, 1536, 17, 2), (5, 3328, 31, 3), (131, 1280, 64, 6), (500, 1280, 40, 2), (500, 512, 100, 4), (257, 256, 241, 8),
                                     (131, 1536, 64, 6), (500, 2048, 40, 2), (500, 1024, 100, 4), (230, 512, 241, 8), (9, 768, 65, 3)])
def test_sums_split_by_experts(T, d, E, K):
    logits_bit_for_bit(T, d, E, K)
