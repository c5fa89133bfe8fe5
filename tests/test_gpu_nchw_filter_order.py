"""Plain NCHW through the packed kernels: the conversion writes the filter in the order of a pre-processed one, without padding its channels.
Channels that fill no block, reductions of one step to many, groups, on the tiles that split the reduction and on the staged ones."""
import pytest

from megengine_amd import _abi
from tests import routes
from tests.gpu_util import check_case

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05, nonline="RELU")
# n, ic, h, w, oc, f, stride, groups; the kernel behind the conversion
CASES = [
    ((3, 33, 17, 19, 5, 7, 1, 1), "ks_kernel<32"),
    ((2, 70, 9, 11, 31, 7, 2, 1), "ks_kernel<32"),
    ((1, 270, 14, 13, 130, 3, 1, 1), "ks_kernel<32"),
    ((1, 333, 8, 27, 97, 5, 2, 1), "ks_kernel<32"),
    ((2, 142, 72, 61, 6, 5, 2, 1), "ks_kernel<32"),       # few channels, many pixels
    ((9, 70, 40, 41, 33, 7, 1, 1), "igemm2_kernel"),      # more than the tiles that split are for
    ((3, 64, 9, 10, 128, 3, 1, 2), "igemm2_kernel"),
]


def _desc(n, ic, h, w, oc, f, s, g, z):
    return _abi.make_conv_desc("NCHW", n, ic, h, w, oc, f, pad=f // 2, stride=s, group=g, has_z=z, **S)


def test_route():
    for (case, kernel), got in zip(CASES, routes.routes([_desc(*case, False) for case, _ in CASES])):
        assert got.kernels[0] == "nchw_prep_kernel" and kernel in got.kernels[1], (case, got.kernels)


@pytest.mark.gpu
@pytest.mark.parametrize("case,kernel", CASES)
def test_filter_order(oracle, case, kernel):
    for z in (False, True):
        assert check_case(oracle, _desc(*case, z), seed=case[1], tag=kernel) is not None
