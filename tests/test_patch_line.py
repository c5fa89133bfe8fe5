"""Dense 3x3 layers over 32 or 64 channels at stride 1 whose filter is pre-processed, from 1200 tiles of 64 x 128 on (no GPU): the
one-stage patch tile or the ring, whichever was faster in graph replays."""
import pytest

from megengine_amd import _abi, lib, ops

# n, ic, h, w, oc, residual; us of both
LAYERS = [
    (42, 32, 50, 25, 160, True, {"dma128x64x128r2": 13.9, "v2_patch_32x256": 9.7}),
    (55, 32, 56, 56, 32, True, {"32x256x128": 13.1, "v2_patch_32x256": 7.9}),
    (62, 64, 56, 56, 32, True, {"32x256x128": 16.3, "v2_patch_32x256": 9.4}),
    (41, 64, 20, 49, 288, True, {"dma128x64x128r2": 19.7, "v2_patch_32x256": 14.0}),
    (30, 64, 30, 77, 160, True, {"dma128x128x128r2w8": 20.6, "v2_patch_32x256": 13.7}),
    (50, 64, 33, 69, 96, True, {"dma128x64x128r2": 18.0, "v2_patch_32x256": 13.8}),
    (39, 64, 61, 20, 288, False, {"v2_128x128x64r4": 16.7, "v2_patch_32x256": 16.3}),
    (16, 32, 56, 56, 288, False, {"v2_128x128x64r4": 13.3, "v2_patch_32x256": 11.5}),
    (74, 32, 45, 79, 32, False, {"v2_64x128x64r4": 12.7, "v2_patch_32x256": 7.9}),
    (18, 64, 56, 56, 288, False, {"v2_128x128x64r4": 20.0, "v2_patch_32x256": 16.5}),
    (116, 64, 24, 27, 224, False, {"v4_64x128res": 23.3, "v2_patch_32x256": 18.2}),
    (38, 32, 62, 69, 96, True, {"v4_64x128res": 19.8, "v2_patch_32x256": 14.6}),
    (49, 32, 56, 56, 64, True, {"dma64x128x128r2": 12.0, "v2_patch_64x256": 10.4}),
    (51, 64, 59, 53, 64, False, {"v2_64x128x64r4": 12.3, "v2_patch_64x256": 12.5}),
    (36, 64, 80, 58, 64, False, {"v2_64x128x64r4": 14.5, "v2_patch_64x256": 12.6}),
    (40, 64, 59, 72, 64, False, {"v2_64x128x64r4": 14.4, "v2_patch_64x256": 12.6}),
    (77, 32, 31, 74, 64, False, {"v2_64x128x64r4": 11.4, "v2_patch_64x256": 10.5}),
    (60, 64, 56, 56, 64, False, {"v2_64x128x64r4": 13.8, "v2_patch_64x256": 13.4}),
]


@pytest.mark.parametrize("i", range(len(LAYERS)))
def test_line(i):
    n, ic, h, w, oc, z, us = LAYERS[i]
    d = _abi.make_conv_desc("NCHW32", n, ic, h, w, oc, 3, pad=1, nonline="RELU", has_z=z, scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
    a, _ = ops.conv_bias_query(d, _abi.ALGO_HEURISTIC_PREPROCESS)
    assert a.id == 1
    # 3 %: what two runs of one tile differ by
    assert us[lib.tile_names()[a.tile_cfg]] <= 1.03 * min(us.values())
