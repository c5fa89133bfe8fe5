"""The vector forms of channel-wise convolution where the matrix form (test_gpu_dw_matrix.py) leaves layers to them: dwf_kernel for many
small planes of 5x5 and 7x7 and where its price is lower, one and two output rows per thread, and dw4_kernel for wide strides of few taps, large windows and rows whose
patch does not fit.  Each case names the kernel that it is about."""
import pytest

from megengine_amd import _abi
from tests.gpu_util import check_case
from tests.routes import routes

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
CASES = [
    # n, channels, ih, iw, fh, fw, pad, stride, kernel
    (16, 128, 7, 7, 5, 5, 2, 1, "dwf_kernel<5, 1, 1>"),        # 512 planes, rows of seven
    (19, 108, 14, 14, 5, 5, 2, 2, "dwf_kernel<5, 2, 1>"),      # 513
    (16, 128, 3, 5, 7, 7, 3, 1, "dwf_kernel<7, 1, 1>"),        # smaller than the filter
    (8, 256, 13, 11, 7, 7, 3, 2, "dwf_kernel<7, 2, 1>"),
    (8, 256, 1, 1, 5, 5, 2, 1, "dwf_kernel<5, 1, 1>"),
    (8, 256, 9, 43, 5, 5, 2, 1, "dwf_kernel<5, 1, 1>"),        # 99 quads
    (8, 256, 10, 38, 5, 5, 2, 1, "dwm_kernel<3, true>"),       # 100
    (7, 292, 9, 43, 5, 5, 2, 1, "dwm_kernel<3, true>"),        # 511 planes
    (32, 256, 24, 15, 5, 5, 2, 1, "dwf_kernel<5, 1, 2>"),      # two rows per thread
    (32, 256, 23, 14, 5, 5, 2, 1, "dwf_kernel<5, 1, 2>"),      # an odd number of them
    (32, 256, 47, 29, 5, 5, 2, 2, "dwf_kernel<5, 2, 2>"),
    (32, 256, 45, 31, 5, 5, 2, 2, "dwf_kernel<5, 2, 2>"),
    (32, 264, 21, 13, 7, 7, 3, 1, "dwf_kernel<7, 1, 2>"),
    (32, 256, 45, 32, 7, 7, 3, 2, "dwf_kernel<7, 2, 2>"),
    (1, 8, 5, 1701, 5, 5, 2, 1, "dwf_kernel<5, 1, 1>"),        # no room for a row's patch
    (7, 172, 18, 40, 5, 5, 2, 1, "dwf_kernel<5, 1, 1>"),       # by price: 301 workgroups of the matrix form on 256 CUs
    (9, 48, 31, 143, 5, 5, 2, 2, "dwf_kernel<5, 2, 1>"),       # its patch is two copies wide
    (2, 12, 44, 41, 7, 1, (3, 0), 3, "dw4_kernel"),
    (2, 12, 23, 46, 2, 4, (1, 2), (1, 3), "dw4_kernel"),
    (2, 8, 31, 33, 5, 5, 2, 5, "dw4_kernel"),
    (1, 8, 31, 30, 11, 11, 5, 1, "dw4_kernel"),
    (2, 8, 23, 27, 10, 9, (12, 4), 2, "dw4_kernel"),           # padding wider than the filter
    (1, 4, 5, 1703, 5, 5, (2, 1), 1, "dw4_kernel"),
    (2, 8, 140, 9, 5, 5, (0, 2), (70, 1), "dw4_kernel"),
    (1, 4, 1, 1, 11, 11, 5, 1, "dw4_kernel"),
    (8, 100, 25, 37, 1, 1, 0, 1, "dw4_kernel"),                # one tap, two at stride 2: more than 40000 quads out
    (10, 100, 49, 125, 2, 1, (1, 0), 2, "dw4_kernel"),
    (10, 100, 51, 123, 1, 2, (0, 1), 2, "dw4_kernel"),
    (8, 100, 25, 32, 1, 1, 0, 1, "dwm_kernel<1, true>"),       # exactly that many
]


def _kernel(d):
    (r,) = routes([d])
    return r.kernels


@pytest.mark.parametrize("i", range(len(CASES)))
def test_vector_forms(oracle, i):
    n, c, ih, iw, fh, fw, pad, stride, kernel = CASES[i]
    conv = lambda **kw: _abi.make_conv_desc("NCHW4", n, c, ih, iw, c, fh, fw, group=c, pad=pad, stride=stride, **kw)  # noqa: E731
    for nl, kw in (("RELU", dict()), ("H_SWISH", dict(has_z=True)), ("IDENTITY", dict(bias_mode=_abi.BIAS_NONE))):
        d0 = conv(nonline=nl, **kw, **S)
        ss, _, _, ds = _abi.conv_shapes(d0)
        si, do = ss[1] * ss[2] * ss[3] * ss[4], ds[1] * ds[2] * ds[3] * ds[4]
        d = conv(nonline=nl, src_stride_n=si + 4, dst_stride_n=do + 8, z_stride_n=do + 12 if "has_z" in kw else 0, **kw, **S)
        for desc in (d0, d):
            assert _kernel(desc) == (kernel if "has_z" in kw else kernel.replace("true", "false"),)
            check_case(oracle, desc, seed=110 + i, tag="dw vector %d" % i)
    # the one-instruction requantisation, and scales outside the range of the divide-free epilogue
    check_case(oracle, conv(nonline="RELU", scale_bias=1.3e-3, scale_dst=0.0271), seed=130 + i, tag="dw vector %d linear" % i)
    check_case(oracle, conv(nonline="RELU", has_z=True, scale_bias=1e-20, scale_z=3e-19, scale_dst=1e-18), seed=150 + i,
               tag="dw vector %d literal" % i)
