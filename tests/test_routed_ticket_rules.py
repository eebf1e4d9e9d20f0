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


# measured: 12 strips by tickets, strips in multiples of 8 only where they are short, long ones and hundreds of rows a group not
@pytest.mark.parametrize("K,strips,pairs,groups,want", [
    (3072, 12, 16384, 256, 1), (3072, 12, 43520, 256, 1), (3072, 12, 76800, 256, 0), (2048, 8, 25600, 256, 1), (2048, 8, 76800, 256, 0), (3072, 8, 33280, 256, 0),
    (3072, 16, 16500, 256, 0), (4096, 8, 16384, 256, 0), (4096, 16, 16500, 256, 0), (3584, 12, 16500, 256, 0), (1536, 12, 25600, 256, 1), (1536, 12, 76800, 256, 0),
    (1024, 8, 25600, 256, 1), (768, 8, 25600, 256, 0), (512, 12, 16384, 256, 0)])
def test_products_that_take_tickets(K, strips, pairs, groups, want):
    from llmx_amd import ops
    assert ops.lib().llmx_tile_takes_tickets(K, strips, pairs, groups) == want


@pytest.mark.parametrize("pairs,n128,n64,experts", [(8192, 256, 256, 256), (16384, 256, 393, 256), (33280, 406, 640, 256), (43520, 512, 780, 256),
                                                    (76800, 766, 1270, 256), (16384, 164, 290, 55), (1000, 8, 16, 8)])
def test_a_product_without_tickets_finds_its_own_choice(pairs, n128, n64, experts):
    from llmx_amd import ops
    got = ops.lib().llmx_tile_choice_tickets(pairs, n128, n64, experts)
    assert (got ^ got >> 4) & 15 == ops.lib().llmx_tile_choice(pairs, n128, n64, experts)
