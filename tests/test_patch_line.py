"""Lines of the one-stage patch tiles for 3x3 layers over 32 or 64 channels (no GPU): dense layers at stride 1 whose filter is
pre-processed, from 1200 tiles of 64 x 128 on, and group layers at stride 2, against the ring: whichever was faster in graph replays."""
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


# n, groups, channels in and out per group, ih, iw; us on the second-generation tiles and on the patch tiles.  Of 3000 drawn group layers the
# strided ones without a residual into more than 64 channels: every 14th that is more than 5 % behind on the patch tiles and every
# 40th that is ahead
GROUPS = [
    (15, 7, 64, 256, 33, 79, 21.1, 23.9),
    (56, 2, 32, 96, 42, 68, 8.9, 9.5),
    (53, 8, 32, 256, 18, 24, 9.6, 10.8),
    (28, 8, 32, 192, 46, 12, 7.8, 9.6),
    (35, 5, 64, 128, 42, 85, 24.0, 26.4),
    (37, 3, 64, 160, 60, 42, 18.1, 19.8),
    (10, 4, 64, 160, 66, 62, 11.5, 12.6),
    (7, 8, 64, 256, 41, 44, 10.0, 11.4),
    (26, 6, 64, 256, 52, 48, 27.7, 33.8),
    (37, 10, 64, 96, 10, 62, 9.1, 12.2),
    (11, 4, 64, 256, 93, 66, 24.3, 27.1),
    (54, 6, 64, 256, 58, 12, 19.3, 25.5),
    (29, 7, 32, 192, 22, 28, 7.3, 8.6),
    (5, 11, 64, 128, 46, 46, 8.8, 10.0),
    (59, 4, 64, 256, 76, 30, 40.9, 49.4),
    (15, 9, 64, 128, 48, 55, 14.7, 16.4),
    (58, 5, 32, 256, 19, 42, 12.3, 13.5),
    (21, 5, 32, 192, 39, 39, 11.1, 11.8),
    (48, 4, 64, 192, 20, 79, 20.9, 22.6),
    (30, 4, 64, 256, 72, 57, 35.7, 42.9),
    (18, 16, 64, 256, 39, 18, 18.9, 20.9),
    (27, 3, 32, 192, 24, 30, 7.3, 6.0),
    (7, 4, 64, 96, 30, 41, 5.6, 4.9),
    (17, 2, 64, 192, 10, 18, 5.2, 3.8),
    (4, 8, 64, 160, 31, 11, 5.2, 4.6),
    (48, 2, 64, 96, 12, 63, 7.2, 5.3),
    (6, 2, 32, 192, 21, 15, 5.2, 4.0),
    (17, 3, 64, 192, 20, 46, 8.1, 6.4),
    (50, 2, 64, 96, 104, 13, 10.1, 8.6),
    (4, 3, 32, 128, 37, 14, 5.1, 3.8),
    (7, 6, 64, 192, 103, 33, 14.0, 12.4),
    (21, 15, 32, 128, 23, 53, 13.8, 12.6),
    (11, 2, 64, 128, 18, 46, 5.2, 4.0),
    (12, 3, 64, 160, 41, 17, 5.6, 5.0),
]


def test_strided_groups():
    lost = []
    for n, g, ic, oc, h, w, ring, patch in GROUPS:
        d = _abi.make_conv_desc("NCHW32", n, ic * g, h, w, oc * g, 3, pad=1, stride=2, group=g, nonline="RELU", scale_bias=2e-4, scale_dst=0.05)
        a, _ = ops.conv_bias_query(d)
        assert a.id == 1
        lost.append((patch if lib.tile_names()[a.tile_cfg].startswith("v2_patch_") else ring) / min(ring, patch) - 1)
    # 7 of these 34 are more than 3 % behind the faster way, at most 23 %; always on the patch tiles 21 are, by up to 34 %
    assert sum(l > 0.03 for l in lost) <= 7 and max(lost) <= 0.24, lost
