"""3x3 layers over at most 64 4-packed channels, whose whole reduction is one stage: channel blocks that do not fill a group of 16 or 32, output
channels that end inside a tile, planes of one pixel and rows wider than a tile, several images in a tile, strides, batch strides."""
import pytest

from megengine_amd import _abi, lib
from tests.gpu_util import check_case
from tests.routes import routes

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
CASES = [
    # n, ic, ih, iw, oc, pad, stride
    (1, 4, 1, 1, 4, 1, 1),
    (9, 16, 7, 7, 20, 1, 1),          # several images in a tile
    (1, 20, 5, 300, 36, 1, 1),        # rows wider than a tile, a second group of channels of one block
    (2, 32, 13, 17, 64, 0, 1),
    (2, 36, 20, 11, 68, 2, 1),        # one block past 32 channels
    (1, 64, 31, 33, 32, 1, 2),
    (2, 60, 29, 18, 100, 1, 2),
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_one_stage(oracle, i):
    n, ic, ih, iw, oc, pad, stride = CASES[i]
    for nl, kw in (("RELU", dict(has_z=True)), ("IDENTITY", dict()), ("H_SWISH", dict(bias_mode=_abi.BIAS_NONE))):
        d0 = _abi.make_conv_desc("NCHW4", n, ic, ih, iw, oc, 3, pad=pad, stride=stride, nonline=nl, **kw, **S)
        ss, _, _, ds = _abi.conv_shapes(d0)
        do = ds[1] * ds[2] * ds[3] * ds[4]
        d1 = _abi.make_conv_desc("NCHW4", n, ic, ih, iw, oc, 3, pad=pad, stride=stride, nonline=nl, src_stride_n=ss[1] * ss[2] * ss[3] * ss[4] + 8,
                                 dst_stride_n=do + 4, z_stride_n=do + 12 if "has_z" in kw else 0, **kw, **S)
        for d in (d0, d1):
            for t in [k for k, name in enumerate(lib.tile_names()) if name.startswith("patch4_")]:
                assert routes([(d, 1, t, False)])[0].kernels[0].startswith("patch4_one_kernel<%d," % (1 if ic <= 32 else 2))
                assert check_case(oracle, d, seed=60 + i, algo=1, tile=t, tag=lib.tile_names()[t]) is not None
