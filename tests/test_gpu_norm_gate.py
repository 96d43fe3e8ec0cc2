"""Block form, forward and backward, at the edges of the row kernels of the norm (two rows per workgroup, one, or rows in
chunks; widths that leave pieces of a thread unused) and of the gate-gradient kernel (experts behind a unit of 32, columns
behind a block of 256, token slices of odd length).  Row statistics bit for bit; gradients within the fp32 (1e-5) and bf16
(1e-2) relative L2 of every layer test."""
import pytest

from tests.test_gpu_block import test_block_backward_matches_oracle as block_backward
from tests.test_gpu_block import test_block_forward_matches_oracle as block_forward

pytestmark = pytest.mark.gpu

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
