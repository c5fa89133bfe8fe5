"""The 4-packed patch tiles (patch4_*) where they can go wrong: channel blocks that do not fill a group of sixteen, an odd
number of groups and of filter entries, output channels and pixels around the edges of a tile, several small images in one
tile, wide rows in several columns, windows that hang over every border, strides, batch strides larger than an image."""
import pytest

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
IGEMM = 1
CASES = [
    # n, ic, ih, iw, oc, f, pad, stride
    (1, 4, 3, 3, 4, 3, 1, 1),          # one channel block, fewer pixels than a wave
    (5, 16, 7, 7, 32, 3, 1, 1),        # one group, several images in a tile, the last one incomplete
    (3, 20, 9, 11, 36, 3, 1, 1),       # two groups, the second of one block; 36 channels
    (2, 52, 13, 17, 100, 3, 0, 1),     # four groups, the last of one block
    (1, 100, 6, 40, 68, 3, 1, 2),      # seven groups: the last stage holds one
    (2, 24, 5, 300, 24, 3, 1, 1),      # rows wider than a tile
    (2, 40, 33, 35, 132, 5, 2, 1),     # 25 taps: an odd number of entries
    (2, 36, 19, 23, 40, 5, 2, 2),
    (1, 16, 12, 15, 20, 7, 3, 1),      # 49 taps: only the 32-channel tiles
    (2, 32, 8, 9, 64, 2, 1, 1),        # even filter
    (1, 12, 1, 65, 8, 3, 1, 1),        # one row
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_every_tile(oracle, i):
    n, ic, ih, iw, oc, f, pad, stride = CASES[i]
    tiles = [t for t, name in enumerate(lib.tile_names()) if name.startswith("patch4_")]
    ran = 0
    for nl, z in (("RELU", True), ("IDENTITY", False), ("H_SWISH", True)):
        d = _abi.make_conv_desc("NCHW4", n, ic, ih, iw, oc, f, pad=pad, stride=stride, nonline=nl, has_z=z, **S)
        for t in tiles:
            if check_case(oracle, d, seed=90 + i, algo=IGEMM, tile=t, tag=lib.tile_names()[t]) is not None:
                ran += 1
    assert ran >= 6
