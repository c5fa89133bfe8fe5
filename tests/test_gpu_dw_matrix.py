"""Channel-wise convolution on the matrix cores, where it can go wrong: quads and blocks that hang over a row's end, bands of rows, narrow
patches with several rows to a copy, patches wider than a wave, strides up to four, paddings wider than the filter, batch strides."""
import pytest

from megengine_amd import _abi, ops
from tests.gpu_util import check_case
from tests.routes import routes

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
DW = 2
CASES = [
    # n, channels, ih, iw, fh, fw, pad, stride
    (1, 4, 1, 1, 5, 5, 2, 1),                # one pixel, one quad
    (2, 12, 5, 3, 5, 5, 2, 1),
    (1, 8, 29, 31, 5, 5, 2, 2),
    (3, 8, 57, 57, 5, 5, 2, 2),
    (1, 4, 90, 61, 7, 7, 3, 1),              # several bands, the last one short; 67 columns
    (2, 4, 17, 130, 7, 7, 3, 2),             # three copies per row
    (1, 4, 3, 1000, 5, 5, 2, 1),             # one row to a band
    (2, 8, 20, 14, 4, 6, (0, 5), (1, 2)),
    (1, 8, 23, 22, 1, 7, (0, 3), 1),
    (1, 8, 23, 22, 7, 1, (3, 0), (2, 1)),
    (2, 8, 12, 13, 2, 2, 0, 1),
    (1, 4, 31, 30, 9, 9, 4, 1),              # seven steps
    (1, 4, 40, 33, 8, 4, 9, 1),              # padding wider than the filter
    (1, 8, 21, 26, 3, 3, 1, (3, 3)),
    (1, 8, 25, 40, 3, 5, 1, (4, 4)),
    (1, 8, 29, 31, 5, 5, (1, 2), (1, 2)),    # the third and the seventh again, as the matrix form takes them
    (1, 4, 3, 1000, 5, 5, (2, 3), 1),
]
VECTOR = (2, 6)  # dwf_kernel is ahead there, at its price


@pytest.mark.parametrize("i", range(len(CASES)))
def test_depthwise_matrix(oracle, i):
    n, c, ih, iw, fh, fw, pad, stride = CASES[i]
    for nl, kw in (("RELU", dict()), ("H_SWISH", dict(has_z=True)), ("IDENTITY", dict(bias_mode=_abi.BIAS_NONE))):
        d0 = _abi.make_conv_desc("NCHW4", n, c, ih, iw, c, fh, fw, group=c, pad=pad, stride=stride, nonline=nl, **kw, **S)
        ss, _, _, ds = _abi.conv_shapes(d0)
        si, do = ss[1] * ss[2] * ss[3] * ss[4], ds[1] * ds[2] * ds[3] * ds[4]
        d = _abi.make_conv_desc("NCHW4", n, c, ih, iw, c, fh, fw, group=c, pad=pad, stride=stride, nonline=nl, src_stride_n=si + 4,
                                dst_stride_n=do + 8, z_stride_n=do + 12 if "has_z" in kw else 0, **kw, **S)
        for desc in (d0, d):
            a, _ = ops.conv_bias_query(desc)
            assert a.id == DW and routes([desc])[0].kernels[0].startswith("dwf_kernel" if i in VECTOR else "dwm_kernel")
            check_case(oracle, desc, seed=50 + i, tag="dw matrix %d" % i)
    # scales outside the range of the divide-free epilogue
    d = _abi.make_conv_desc("NCHW4", n, c, ih, iw, c, fh, fw, group=c, pad=pad, stride=stride, nonline="RELU", has_z=True,
                            scale_bias=1e-20, scale_z=3e-19, scale_dst=1e-18)
    check_case(oracle, d, seed=80 + i, tag="dw matrix %d literal" % i)
