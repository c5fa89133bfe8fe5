"""Channel-wise 5x5 and 7x7 convolutions at widths around the blocks of four pixels, odd heights, images smaller than the filter,
both strides, every activation with and without a residual, and other paddings and strides: on these few or large planes all of them but one
run the matrix form (test_gpu_dw_matrix.py); the vector forms have their cases in test_gpu_dw_vector.py.  3x3 layers with one,
two and four output rows per thread."""
import pytest

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)


@pytest.mark.parametrize("f", [5, 7])
@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("ih,iw", [(1, 1), (3, 2), (5, 4), (6, 5), (8, 7), (9, 8), (7, 13), (12, 16), (11, 33)])
def test_same_padding(oracle, f, stride, ih, iw):
    for k, (nl, z, c) in enumerate((("RELU", False, 8), ("IDENTITY", True, 4), ("H_SWISH", False, 12))):
        d = _abi.make_conv_desc("NCHW4", 3, c, ih, iw, c, f, pad=f // 2, stride=stride, group=c, nonline=nl, has_z=z, **S)
        assert lib.algo_names()[ops.conv_bias_query(d)[0].id] == "MI355_DEPTHWISE_DOT4"
        check_case(oracle, d, seed=10 * f + stride + k, tag="dw%d" % f)
    # scales for which the one-instruction requantisation is proved
    d = _abi.make_conv_desc("NCHW44", 2, 8, ih, iw, 8, f, pad=f // 2, stride=stride, group=8, nonline="RELU", scale_bias=1.3e-3,
                            scale_dst=0.0271)
    check_case(oracle, d, seed=f, tag="dw%d linear" % f)


@pytest.mark.parametrize("f,pad,stride", [(5, 0, 1), (5, (2, 1), 1), (7, 4, 2), (5, 2, 3)])
def test_other_paddings_and_strides(oracle, f, pad, stride):
    d = _abi.make_conv_desc("NCHW4", 2, 8, 11, 13, 8, f, pad=pad, stride=stride, group=8, nonline="RELU", has_z=True, **S)
    check_case(oracle, d, seed=5, tag="dw other")


def test_height_padding_may_differ(oracle):
    d = _abi.make_conv_desc("NCHW4", 2, 8, 11, 13, 8, 5, pad=(1, 2), stride=1, group=8, nonline="RELU", **S)
    check_case(oracle, d, seed=6, tag="dw pad_h 1")


@pytest.mark.parametrize("n,c,ih,iw,f,stride", [
    (40, 64, 41, 37, 3, 1),   # two output rows per thread, an odd number of them
    (40, 64, 41, 37, 5, 1),
    (40, 64, 81, 73, 5, 2),
    (41, 64, 43, 33, 7, 1),
    (64, 96, 44, 59, 3, 1),   # four
    (40, 64, 81, 75, 3, 2),   # one at any size
    (64, 640, 7, 7, 3, 1),    # planes of seven rows, around the line between one and two
    (64, 736, 7, 6, 3, 1),
])
def test_rows_per_thread(oracle, n, c, ih, iw, f, stride):
    """(the lines of 5x5 and 7x7 are the matrix form's now: large planes, several bands)"""
    for nl, z in (("RELU", False), ("IDENTITY", True)):
        d = _abi.make_conv_desc("NCHW4", n, c, ih, iw, c, f, pad=f // 2, stride=stride, group=c, nonline=nl, has_z=z, **S)
        check_case(oracle, d, seed=70 + f, tag="dw rows")
