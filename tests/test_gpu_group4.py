"""NCHW4 group convolutions in one launch (tile grp4_dot4) at the edges of its threads' work: odd output heights (a thread
makes two rows of a 3x3 layer), column counts around a workgroup, strides, filters other than 3x3, channel quads that do
and do not pair up, batch-strided views; against the checker, and equal to one dense launch per group."""
import numpy as np
import pytest

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
IGEMM = 1
CASES = [
    # n, groups, icpg, ocpg, ih, iw, f, pad, stride
    (1, 2, 4, 4, 1, 1, 3, 1, 1),
    (2, 3, 4, 4, 7, 9, 3, 1, 1),
    (2, 4, 8, 8, 16, 32, 3, 1, 1),     # exactly one workgroup of columns and row pairs
    (1, 5, 12, 4, 17, 31, 3, 1, 1),
    (2, 2, 16, 16, 9, 8, 3, 0, 1),
    (1, 3, 8, 24, 11, 13, 3, 1, 2),
    (2, 2, 4, 12, 12, 10, 3, 2, 2),
    (1, 4, 16, 8, 6, 7, 5, 2, 1),
    (2, 2, 8, 4, 5, 5, 1, 0, 1),
    (1, 2, 4, 8, 9, 9, 3, 1, 3),
    # whole slabs of 16 channels: bands of rows on the matrix cores
    (1, 4, 4, 4, 3, 338, 3, 1, 1),     # one row per band
    (1, 4, 4, 4, 3, 340, 3, 1, 1),     # a row does not fit: dot products
    (3, 8, 4, 4, 23, 30, 3, 1, 1),     # several bands, the last one incomplete
    (2, 4, 8, 8, 21, 35, 3, 1, 2),
    (2, 3, 16, 16, 40, 25, 3, 2, 1),
    (1, 4, 8, 8, 2, 2, 3, 1, 1),
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_one_launch_for_all_groups(oracle, i):
    n, g, icpg, ocpg, ih, iw, f, pad, stride = CASES[i]
    names = lib.tile_names()
    for nl, z in (("RELU", True), ("IDENTITY", False), ("H_SWISH", False)):
        kw = dict(pad=pad, stride=stride, group=g, nonline=nl, has_z=z, **S)
        d = _abi.make_conv_desc("NCHW4", n, g * icpg, ih, iw, g * ocpg, f, **kw)
        algo, _ = ops.conv_bias_query(d)
        assert algo.id == IGEMM and names[algo.tile_cfg] == "grp4_dot4"
        check_case(oracle, d, seed=20 + i, tag="grp4 %d" % i)
        check_case(oracle, d, seed=20 + i, algo=IGEMM, tile=names.index("64x64x128"), tag="per group %d" % i)
        ss, _, _, ds = _abi.conv_shapes(d)
        d = _abi.make_conv_desc("NCHW4", n, g * icpg, ih, iw, g * ocpg, f, src_stride_n=int(np.prod(ss[1:])) + 32,
                                dst_stride_n=int(np.prod(ds[1:])) + 16, z_stride_n=int(np.prod(ds[1:])) + 48, **kw)
        check_case(oracle, d, seed=40 + i, tag="grp4 strided %d" % i)


def test_wide_groups_keep_a_launch_of_matrix_tiles_each():
    d = _abi.make_conv_desc("NCHW4", 1, 64, 8, 8, 64, 3, pad=1, group=2, **S)
    algo, _ = ops.conv_bias_query(d)
    assert algo.id == IGEMM and lib.tile_names()[algo.tile_cfg] != "grp4_dot4"


@pytest.mark.parametrize("case", [(1, 2, 16, 32, 20, 20, (7, 7), 1), (3, 2, 16, 20, 19, 33, (5, 5), 2), (6, 2, 8, 36, 30, 36, (3, 6), 1),
                                  (2, 2, 16, 8, 40, 11, (18, 1), 1)])
def test_groups_with_many_taps_run_group_by_group(oracle, case):
    """Where the default is a dense launch per group: its results, residuals and batch strides."""
    n, g, icpg, ocpg, ih, iw, f, stride = case
    names = lib.tile_names()
    for nl, z in (("RELU", True), ("IDENTITY", False), ("H_SWISH", True)):
        kw = dict(pad=(f[0] // 2, f[1] // 2), stride=stride, group=g, nonline=nl, has_z=z, **S)
        d = _abi.make_conv_desc("NCHW4", n, g * icpg, ih, iw, g * ocpg, *f, **kw)
        algo, _ = ops.conv_bias_query(d)
        assert algo.id == IGEMM and names[algo.tile_cfg] != "grp4_dot4"
        check_case(oracle, d, seed=60 + icpg, tag="default " + names[algo.tile_cfg])
        check_case(oracle, d, seed=60 + icpg, algo=IGEMM, tile=names.index("grp4_dot4"), tag="one launch")
        ss, _, _, ds = _abi.conv_shapes(d)
        d = _abi.make_conv_desc("NCHW4", n, g * icpg, ih, iw, g * ocpg, *f, src_stride_n=int(np.prod(ss[1:])) + 32,
                                dst_stride_n=int(np.prod(ds[1:])) + 16, z_stride_n=int(np.prod(ds[1:])) + 48, **kw)
        check_case(oracle, d, seed=80 + icpg, tag="default strided")
