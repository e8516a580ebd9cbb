"""The stand-alone step's tiling setting: saving it, changing it and setting it back leaves the
choice by the grid's size in force (no GPU needed: the setting is the host's)."""
from asteriy_2d_amd import native


def test_save_and_restore_keeps_the_choice_by_size():
    L = native.load()
    setting = getattr(L, "_Z21ast_tile_rows_settingv")  # what a step goes by; 0: the grid's size
    old = L.ast_get_tile_rows()
    try:
        assert L.ast_set_tile_rows(8) == 0 and setting() == 0
        saved = L.ast_get_tile_rows()
        for tile in (6, -12, 16):
            assert L.ast_set_tile_rows(tile) == 0
            assert L.ast_get_tile_rows() == tile and setting() == tile
        assert L.ast_set_tile_rows(saved) == 0 and setting() == 0
        for bad in (0, 1025, -(1 << 20) - 1):
            assert L.ast_set_tile_rows(bad) != 0 and setting() == 0
    finally:
        L.ast_set_tile_rows(old)
