"""The tiles that split the reduction over the waves of a workgroup (v2_ks_*, ks4_*) where they can go wrong: reductions
with fewer steps than waves, an odd number of 32-byte chunks, rows that end inside a chunk, pixels and channels around the
16 / 32 / 64 of a tile, more tiles than the eight XCDs and fewer, windows that hang over every border."""
import numpy as np
import pytest

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
IGEMM = 1
CASES = [
    # fmt, n, ic, ih, iw, oc, f, pad, stride
    ("NCHW32", 1, 32, 1, 1, 32, 1, 0, 1),          # one pixel, one step
    ("NCHW32", 1, 96, 7, 7, 64, 1, 0, 1),          # three chunks: an odd number
    ("NCHW32", 1, 32, 5, 7, 96, 3, 1, 1),          # nine chunks, 35 pixels
    ("NCHW32", 2, 64, 9, 3, 288, 3, 1, 2),         # nine channel tiles of 32, strided
    ("NCHW32", 1, 288, 4, 8, 544, 5, 2, 1),        # long reduction, 17 channel blocks
    ("NCHW32", 3, 512, 7, 7, 512, 3, 1, 1),
    ("NCHW32_NCHW4", 1, 64, 6, 6, 20, 3, 1, 1),    # 32-packed in, 4-packed out, 20 channels
    ("NCHW4_NCHW32", 1, 20, 6, 6, 64, 3, 1, 1),
    ("NCHW4", 1, 4, 17, 1, 4, 1, 0, 1),            # one unit of four bytes
    ("NCHW4", 2, 20, 3, 11, 36, 1, 0, 1),          # a row ends inside its chunk
    ("NCHW4", 1, 52, 9, 9, 100, 3, 1, 1),          # 117 units, 15 chunks: odd, the last one incomplete
    ("NCHW4", 1, 200, 5, 5, 28, 5, 2, 2),
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_every_tile(oracle, i):
    fmt, n, ic, ih, iw, oc, f, pad, stride = CASES[i]
    tiles = [t for t, name in enumerate(lib.tile_names()) if name.startswith(("v2_ks_", "ks4_"))]
    ran = 0
    for nl, z in (("RELU", True), ("IDENTITY", False), ("H_SWISH", True)):
        if z and fmt in ("NCHW4_NCHW32", "NCHW32_NCHW4"):
            continue
        d = _abi.make_conv_desc(fmt, n, ic, ih, iw, oc, f, pad=pad, stride=stride, nonline=nl, has_z=z, **S)
        for t in tiles:
            if check_case(oracle, d, seed=60 + i, algo=IGEMM, tile=t, tag=lib.tile_names()[t]) is not None:
                ran += 1
    assert ran >= 6


def test_the_chooser_takes_them_for_few_pixels_only():
    for fmt, ic, hw, oc, f in (("NCHW32", 512, 7, 512, 3), ("NCHW32", 1024, 14, 256, 1), ("NCHW4", 128, 28, 128, 3)):
        names = [lib.tile_names()[ops.conv_bias_query(_abi.make_conv_desc(fmt, n, ic, hw, hw, oc, f, pad=f // 2, **S))[0].tile_cfg]
                 for n in (1, 64)]
        assert "ks" in names[0] and "ks" not in names[1], names


@pytest.mark.parametrize("fh,fw", [(3, 6), (9, 2), (1, 18), (1, 9), (5, 1)])
@pytest.mark.parametrize("fmt,ic,oc", [("NCHW32", 96, 64), ("NCHW4", 20, 36), ("NCHW4_NCHW32", 12, 32), ("NCHW32_NCHW4", 32, 20)])
def test_filters_that_are_not_square(oracle, fmt, ic, oc, fh, fw):
    ran = 0
    for stride in ((1, 1), (2, 1)):
        d = _abi.make_conv_desc(fmt, 2, ic, 11, 19, oc, fh, fw, pad=(fh // 2, fw // 2), stride=stride, nonline="RELU", has_z="_" not in fmt, **S)
        for t, name in enumerate(lib.tile_names()):
            if name.startswith(("v2_ks_", "ks4_")) and check_case(oracle, d, seed=fh + fw, algo=IGEMM, tile=t, tag=name) is not None:
                ran += 1
    assert ran >= 8
