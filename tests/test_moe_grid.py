"""The launch of the experts' tiles: every item has a workgroup, and no dimension holds more threads than the hardware counts."""

import ctypes

import pytest

from nanospec_amd.kernels import build

THREADS = 512  # of a workgroup, at most


@pytest.mark.parametrize("items", [1, 7, 8, 9, 524287, 524288, 524289, (1 << 23) - 8, 1 << 23, (1 << 23) + 1, 65535 * 512, 1 << 30])
def test_the_launch_holds_all_items(items):
    xy = (ctypes.c_uint * 2)()
    build.core().ns_moe_tile_grid(ctypes.c_longlong(items), xy)
    x, y = xy
    assert x % 8 == 0 and items <= x * y < 2 * items + 8  # (an eighth of the items for every XCD)
    assert x * THREADS < 1 << 32 and y <= 65535
