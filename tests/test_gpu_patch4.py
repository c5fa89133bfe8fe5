"""The 4-packed patch tiles (patch4_*) where they can go wrong: channel blocks that do not fill a group of sixteen, an odd
number of groups and of filter entries, output channels and pixels around the edges of a tile, several small images in one
tile, wide rows in several columns, windows that hang over every border, strides, batch strides larger than an image.  3x3 over at most 64
channels is a kernel of its own (test_gpu_patch4_one.py): here, 3x3 over more, in two or more stages, has cases of its own."""
import pytest

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case
from tests.routes import routes

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


# filters that are not square: as many taps as the 3x3 kernel has entries per stage (18: one group of eighteen taps, not two of
# nine), as many as its taps in another arrangement (9), and windows of a single row or column
TAPS = [(3, 6), (6, 3), (2, 9), (9, 2), (1, 18), (18, 1), (1, 9), (9, 1), (1, 7), (2, 5)]


@pytest.mark.parametrize("ic", [8, 16, 20, 52, 100])
@pytest.mark.parametrize("fh,fw", TAPS)
def test_filters_that_are_not_square(oracle, fh, fw, ic):
    tiles = [t for t, name in enumerate(lib.tile_names()) if name.startswith("patch4_")]
    ran = 0
    for oc, stride, z in ((36, 1, True), (68, 2, False)):
        d = _abi.make_conv_desc("NCHW4", 2, ic, 19, 23, oc, fh, fw, pad=(fh // 2, fw // 2), stride=stride, nonline="RELU", has_z=z, **S)
        for t in tiles:
            if check_case(oracle, d, seed=fh * 100 + fw + ic, algo=IGEMM, tile=t, tag=lib.tile_names()[t]) is not None:
                ran += 1
    assert ran >= 4


@pytest.mark.parametrize("fh,fw", [(3, 6), (9, 2), (1, 9)])
def test_filters_that_are_not_square_group_by_group(oracle, fh, fw):
    """Groups of more than sixteen channels run as one dense launch each, on views with the batch strides of the whole."""
    for t, name in enumerate(lib.tile_names()):
        if not name.startswith("patch4_"):
            continue
        d = _abi.make_conv_desc("NCHW4", 3, 40, 13, 18, 72, fh, fw, pad=(fh // 2, fw // 2), group=2, nonline="RELU", has_z=True, **S)
        assert check_case(oracle, d, seed=fh + fw, algo=IGEMM, tile=t, tag=name) is not None


STAGES = [
    # 3x3 over more than 64 channels, two groups of 16 to a stage: n, ic, ih, iw, oc, pad, stride
    (5, 68, 7, 7, 32, 1, 1),          # three stages, the last one of one block; several images in a tile, the last one incomplete
    (3, 80, 9, 11, 36, 1, 1),         # the last one of one group; 36 channels
    (2, 96, 20, 11, 68, 2, 1),        # three whole stages; a window outside the image
    (2, 100, 13, 17, 100, 0, 1),      # four, the last one of one block
    (2, 128, 5, 300, 24, 1, 1),       # four whole ones; rows wider than a tile
    (1, 132, 1, 65, 8, 1, 1),         # five; one row
    (1, 68, 1, 1, 4, 1, 1),
    (2, 72, 29, 18, 100, 1, 2),
    (1, 132, 31, 33, 64, 1, (2, 1)),
]


@pytest.mark.parametrize("i", range(len(STAGES)))
def test_several_stages(oracle, i):
    n, ic, ih, iw, oc, pad, stride = STAGES[i]
    tiles = {t: name for t, name in enumerate(lib.tile_names()) if name.startswith("patch4_")}
    for nl, kw in (("RELU", dict(has_z=True)), ("IDENTITY", dict()), ("H_SWISH", dict(bias_mode=_abi.BIAS_NONE))):
        conv = lambda **more: _abi.make_conv_desc("NCHW4", n, ic, ih, iw, oc, 3, pad=pad, stride=stride, nonline=nl, **kw, **more, **S)  # noqa: E731
        d0 = conv()
        ss, _, _, ds = _abi.conv_shapes(d0)
        do = ds[1] * ds[2] * ds[3] * ds[4]
        d1 = conv(src_stride_n=ss[1] * ss[2] * ss[3] * ss[4] + 8, dst_stride_n=do + 4, z_stride_n=do + 12 if "has_z" in kw else 0)
        for d in (d0, d1):
            kernels = [r.kernels for r in routes([(d, IGEMM, t, False) for t in tiles])]
            assert kernels == [("patch4_kernel<%d, %d, 9>" % tile,) for tile in ((1, 1), (1, 2), (2, 2))]
            for t, name in tiles.items():
                assert check_case(oracle, d, seed=120 + i, algo=IGEMM, tile=t, tag=name) is not None
