"""The tile for a dense 32-packed layer whose filter is in the reference layout (no GPU).  The layers are every fifteenth of the 306 (of
2640 timed) on which prices by launches, rounds and tiles alone, without the terms that TilePrice explains, chose a tile more
than 3 % behind thresholds on tile counts: 1.08 times the best of the six tiles below on average, up to 1.21."""
import math

from megengine_amd import _abi, lib, ops

TILES = ("dma64x128x128w8", "v2_128x256x64r3w8", "v2_64x64x128r4", "dma128x128x128r2w8", "v2_64x128x64r4", "dma64x64x128r4")
# n, ic, h, w, oc, f, stride, residual; us on each of TILES, graph replays on 256 CUs
LAYERS = [
    (10, 768, 14, 30, 544, 3, 2, True, (20.3, 61.7, 22.9, 35.2, 30.1, 19.0)),
    (21, 896, 25, 17, 224, 3, 2, True, (22.7, 61.7, 25.8, 33.6, 32.4, 21.9)),
    (5, 512, 23, 29, 832, 3, 2, True, (15.0, 37.1, 16.8, 24.2, 21.5, 14.6)),
    (3, 384, 15, 70, 736, 3, 2, False, (11.7, 27.8, 12.8, 16.3, 15.9, 11.5)),
    (4, 576, 40, 57, 1024, 3, 2, True, (28.6, 48.1, 40.5, 32.3, 38.2, 33.1)),
    (50, 512, 9, 23, 256, 5, 1, True, (51.1, 85.2, 85.9, 56.9, 72.5, 62.2)),
    (8, 512, 58, 54, 96, 3, 2, True, (14.7, 33.8, 16.5, 20.4, 20.4, 15.0)),
    (4, 64, 12, 68, 640, 5, 1, False, (11.6, 12.6, 10.3, 10.9, 11.6, 9.8)),
    (18, 768, 79, 31, 288, 1, 1, True, (22.7, 29.3, 33.3, 23.1, 25.0, 30.6)),
    (22, 32, 12, 31, 224, 5, 1, False, (6.7, 8.7, 7.3, 7.6, 7.0, 7.1)),
    (15, 512, 91, 97, 64, 1, 1, False, (14.9, 18.5, 16.9, 16.3, 15.6, 14.8)),
    (4, 992, 11, 102, 800, 3, 1, False, (47.5, 56.6, 75.8, 50.3, 54.9, 62.6)),
    (1, 1024, 63, 51, 160, 5, 1, False, (59.9, 162.1, 60.6, 109.8, 81.8, 57.5)),
    (15, 1024, 13, 15, 288, 5, 1, True, (61.3, 164.0, 60.2, 110.4, 82.2, 57.2)),
    (37, 512, 57, 26, 320, 1, 2, False, (9.1, 9.2, 11.6, 8.1, 10.6, 10.0)),
    (17, 768, 16, 17, 160, 5, 1, True, (46.3, 113.9, 46.2, 72.3, 61.3, 44.3)),
    (11, 1024, 18, 32, 96, 5, 1, True, (58.9, 145.5, 60.3, 105.7, 79.6, 57.9)),
    (52, 384, 18, 26, 96, 1, 2, False, (4.9, 6.8, 4.7, 5.1, 5.0, 4.7)),
    (3, 1024, 26, 9, 768, 3, 1, True, (25.6, 61.0, 25.3, 45.0, 33.9, 24.5)),
    (4, 512, 101, 11, 96, 5, 1, False, (31.7, 60.9, 32.0, 47.7, 41.9, 31.0)),
]


def test_lost_layers_are_back():
    ratios = []
    for n, ic, h, w, oc, f, stride, z, us in LAYERS:
        d = _abi.make_conv_desc("NCHW32", n, ic, h, w, oc, f, pad=f // 2, stride=stride, nonline="RELU", has_z=z, scale_bias=2e-4,
                                scale_z=0.05, scale_dst=0.05)
        a, _ = ops.conv_bias_query(d)
        assert a.id == 1
        ratios.append(us[TILES.index(lib.tile_names()[a.tile_cfg])] / min(us))
    mean = math.exp(sum(math.log(r) for r in ratios) / len(ratios))
    # the fit leaves 1.019 on average over all layers and 1.19 at most
    assert mean <= 1.04 and max(ratios) <= 1.2, (mean, ["%.2f" % r for r in ratios])
