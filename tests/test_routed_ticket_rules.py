"""The choice between tiles of 128 and of 64 rows for products that take tiles by tickets, at measured points (classes of K as in the choice without)."""

import pytest


@pytest.mark.parametrize("pairs,n128,n64,experts,want", [
    (8192, 256, 256, 256, 7), (13312, 256, 266, 256, 7), (16384, 256, 393, 256, 7), (25600, 256, 511, 256, 15),      # up to 100 rows an expert
    (33280, 406, 640, 256, 7), (43520, 512, 780, 256, 4), (76800, 766, 1270, 256, None), (16384, 164, 290, 55, 15)])
def test_tiles_chosen(pairs, n128, n64, experts, want):
    from llmx_amd import ops
    got, without = ops.lib().llmx_tile_choice_tickets(pairs, n128, n64, experts), ops.lib().llmx_tile_choice(pairs, n128, n64, experts)
    assert got & without == without and (got & 8) == (without & 8)
    if want is None:
        assert got == without
    else:
        assert got & 7 == want & 7
