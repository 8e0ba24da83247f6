"""Where the fused network runs row by row (ddx_conv_net_rows, host only)."""

import ctypes

import pytest

NET = (3, 32, 32, 32, 32, 2)


def rows(B, H, W, chans=NET):
    from dedalus import _hip
    lib = _hip.load_library()
    return lib.ddx_conv_net_rows(B, H, W, len(chans) - 1, (ctypes.c_int * len(chans))(*chans))


# measured faster row by row: one strip per image and several, 16-row images,
# 32-wide images alone and two to a CU
@pytest.mark.parametrize("B,H,W,S", [(256, 64, 64, 64), (128, 64, 64, 32), (400, 16, 64, 16), (50, 128, 64, 26),
                                     (600, 64, 32, 32), (25, 512, 32, 64), (300, 16, 32, 16), (1024, 32, 32, 32)])
def test_row_by_row(B, H, W, S):
    assert rows(B, H, W) == S


# measured faster on tiles: short strips in several rounds (1150 images 16 x
# 64: 220 us row by row, 203 on tiles), 32-wide strips that just fill the chip
@pytest.mark.parametrize("B,H,W", [(1100, 16, 64), (1150, 16, 64), (300, 32, 64), (275, 32, 64), (128, 64, 32),
                                   (256, 32, 32), (85, 96, 32), (32, 64, 64), (1, 64, 64)])
def test_on_tiles(B, H, W):
    assert rows(B, H, W) == 0


def test_refused():
    assert rows(256, 64, 128) == 0 and rows(256, 72, 64) == 0 and rows(256, 64, 48) == 0
    assert rows(0, 64, 64) == 0 and rows(256, 64, 64, (3, 32, 32, 32, 2)) == 0
    assert rows(256, 64, 64, (3, 16, 16, 16, 16, 2)) == 0 and rows(256, 64, 64, (3, 32, 32, 16, 32, 2)) == 0
