"""fp32 products at row tiles of every height: the checks of test_gpu_f32_products.py on shapes of which it is asserted which height they get, so that another
estimate of the heights cannot move them to other kernels unseen (256 compute units)."""
import pytest

from tests import test_gpu_f32_products as products
from tests.test_gpu_f32_split_range import _height

pytestmark = pytest.mark.gpu

ROWS_128 = dict(T=2708, d=96, H=392, E=3, K=2, Es=1)

CASES = [
    (dict(T=127, d=260, H=132, E=2, K=2), 32),      # whole and partial k steps
    (dict(ROWS_128, H=391), 128),                   # 16-byte loads in the up product alone
    (dict(ROWS_128, d=95), 128),                    # in the down product alone
    (ROWS_128, 128),
    (dict(ROWS_128, d=93, H=391), 128),             # without 16-byte loads
    (products.ROWS_64, 64),
    (dict(products.ROWS_64, d=99, H=131), 64),
]


@pytest.mark.parametrize("kw,rows", CASES)
def test_products_match_oracle_at_their_height(kw, rows):
    assert _height(kw) == rows
    products.test_fp32_products_match_oracle(kw)


@pytest.mark.parametrize("check", [products.test_fp32_training_mode_keeps_h1_h3, products.test_rows_that_start_off_a_16_byte_boundary])
def test_tall_tiles_keep_and_load(check):
    assert _height(ROWS_128) == 128
    check(ROWS_128)


@pytest.mark.parametrize("training", [False, True])
def test_one_layer_at_three_heights(training, monkeypatch):
    assert [_height(dict(ROWS_128, T=T)) for T in (ROWS_128["T"], 900, 77, 1)] == [128, 64, 32, 32]
    monkeypatch.setattr(products, "ROWS_128", ROWS_128)
    products.test_one_layer_at_every_tile_height(training)


@pytest.mark.parametrize("T,d,H,rows", [(64, 64, 3584, 32), (64, 63, 3551, 32), (4096, 96, 3596, 64), (49088, 128, 3584, 128), (49088, 128, 3620, 128)])
def test_two_sums_are_of_every_height(T, d, H, rows):
    """The shapes of products.test_input_gradient_adds_two_sums."""
    assert _height(dict(T=T, d=d, H=H, E=1, K=1)) == rows


@pytest.mark.parametrize("T,d,H,E,rows,cut", [
    (5377, 388, 464, 3, 128, "up down d(a)"), (5505, 395, 463, 3, 128, "up down d(a)"), (4353, 304, 200, 3, 64, "up down"), (4353, 303, 199, 3, 64, "up down"),
    (5529, 256, 516, 2, 64, "up d(a)"), (5529, 256, 515, 2, 64, "up d(a)")])
def test_last_round_in_parts(T, d, H, E, rows, cut):
    """An eighth of the tiles is a whole number of rounds of what an XCD holds and up to 3/8 more (1/4 for 64 x 64 on fp32 MFMAs), which goes in parts of
    32 x 32: with and without 16-byte loads, a single row in an expert's last tile.  The input gradient has the down product's tiles.  Every token goes to
    every expert, so the tiles are known."""
    assert _height(dict(T=T, d=d, H=H, E=E, K=E)) == rows

    def rest(width, columns, slots):
        per = -(-E * -(-T // rows) * -(-columns // width) // 8)
        return per >= slots and 0 < per % slots <= (slots // 4 if slots == 128 else slots * 3 // 8)

    split = 64 if rows == 128 else 96
    got = {"up": rest(64, H, split), "down": rest(128, d, 64) if rows == 128 else rest(64, d, 128), "d(a)": rest(128, H, split)}
    assert " ".join(k for k, v in got.items() if v) == cut
    products.test_last_round_of_tiles_in_parts(T, d, H, E)
