"""RELU without a residual where the scales allow no divide-free form, in the kernels that requantise two dwords at a time (requant8): the
literal chain, not the quotient form with constants that were never made.  Against the oracle."""
import pytest

from megengine_amd import _abi
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu

S = dict(nonline="RELU", scale_bias=1e-20, scale_dst=1e-18)


@pytest.mark.parametrize("gap", [0, 32])   # between images: the kernel's wide argument
@pytest.mark.parametrize("n,c,h,w,f,group", [(2, 8, 23, 22, 7, 8), (2, 32, 11, 13, 3, 8)])
def test_literal_chain(oracle, n, c, h, w, f, group, gap):
    d = _abi.make_conv_desc("NCHW4", n, c, h, w, c, f, pad=f // 2, group=group, src_stride_n=c * h * w + gap if gap else 0, **S)
    check_case(oracle, d, seed=f, tag="literal")
