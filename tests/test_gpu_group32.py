"""The tiles that take the whole reduction of a 3x3 layer over 32 or 64 channels per group in one stage (v2_patch_*), where they can
go wrong: pixels around the edges of a tile, several small images in one, wide rows in several columns, channels that do not fill
a tile of 64, windows that hang over every border, strides, paddings, batch strides; and the choice, which takes them for groups
and dense layers alike."""
import pytest

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
IGEMM = 1
CASES = [
    # n, icpg, ocpg, groups, ih, iw, pad, stride
    (1, 32, 32, 2, 3, 3, 1, 1),
    (9, 32, 32, 3, 7, 7, 1, 1),          # several images in a tile, the last one incomplete
    (2, 64, 64, 2, 13, 17, 0, 1),
    (1, 32, 64, 2, 5, 300, 1, 1),        # rows wider than a tile
    (3, 64, 96, 2, 20, 11, 1, 1),        # a tile of 64 channels half past the group
    (2, 32, 160, 1, 16, 16, 2, 1),       # dense, padding wider than the filter's reach
    (2, 64, 32, 3, 31, 33, 1, 2),
    (1, 32, 64, 2, 29, 64, 0, 3),
    (2, 64, 128, 1, 1, 65, 1, 1),        # one row
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_every_tile(oracle, i):
    n, icpg, ocpg, g, ih, iw, pad, stride = CASES[i]
    tiles = [t for t, name in enumerate(lib.tile_names()) if name.startswith("v2_patch_")]
    ran = 0
    for nl, kw in (("RELU", dict(has_z=True)), ("IDENTITY", dict()), ("H_SWISH", dict(has_z=True, bias_mode=_abi.BIAS_NONE))):
        d = _abi.make_conv_desc("NCHW32", n, icpg * g, ih, iw, ocpg * g, 3, pad=pad, stride=stride, group=g, nonline=nl, **kw, **S)
        for t in tiles:
            if check_case(oracle, d, seed=70 + i, algo=IGEMM, tile=t, tag=lib.tile_names()[t]) is not None:
                ran += 1
    assert ran >= (6 if ocpg == 32 else 9)


def test_batch_strides(oracle):
    d0 = _abi.make_conv_desc("NCHW32", 3, 64, 9, 10, 64, 3, pad=1, group=2, **S)
    _, _, _, ds = _abi.conv_shapes(d0)
    img = ds[1] * ds[2] * ds[3] * ds[4]
    d = _abi.make_conv_desc("NCHW32", 3, 64, 9, 10, 64, 3, pad=1, group=2, nonline="RELU", has_z=True, src_stride_n=img + 32,
                            dst_stride_n=img + 64, z_stride_n=img + 96, **S)
    for t, name in enumerate(lib.tile_names()):
        if name.startswith("v2_patch_32"):
            check_case(oracle, d, seed=7, algo=IGEMM, tile=t, tag=name)


@pytest.mark.parametrize("n,icpg,ocpg,g,hw,stride", [(2, 32, 32, 4, 14, 1), (14, 32, 32, 6, 40, 1), (6, 64, 64, 4, 28, 2), (9, 64, 64, 8, 40, 1),
                                                     (24, 64, 64, 8, 44, 1), (10, 64, 96, 1, 40, 1)])
def test_choice(oracle, n, icpg, ocpg, g, hw, stride):
    d = _abi.make_conv_desc("NCHW32", n, icpg * g, hw, hw, ocpg * g, 3, pad=1, stride=stride, group=g, nonline="RELU", **S)
    a, _ = ops.conv_bias_query(d)
    assert a.id == IGEMM and lib.tile_names()[a.tile_cfg].startswith("v2_patch_")
    check_case(oracle, d, seed=n, tag="choice")
