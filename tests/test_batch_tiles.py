"""Stored lines tiles of the batched loop: "or_planes" leaves to the library whether
rows and lines run together."""
from conftest import pkg


def test_lines_tile_of_a_stored_choice():
    bm = pkg("Programs.find_HII_bubbles_batched")
    assert bm._tile_lines({}) == -1
    assert bm._tile_lines({"columns": 1, "lines": 2}) == 2
    assert bm._tile_lines({"columns": 1, "lines": 2, "or_planes": True}) == -4
    assert bm._tile_lines({"lines": 0, "or_planes": True}) == -2
    for v in bm.load_tiles().values():  # the shipped ones are tuned on neutral boxes
        assert bm._tile_lines(v) <= -2 and v["chosen"][1] != "planes"
