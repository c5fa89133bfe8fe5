"""The bare int32 sums of the staged tiles, whose lanes exchange quads before they store: pixels that end inside a group of four lanes, channels
that end inside a tile, a window and a pointwise layer, batch strides."""
import pytest

from megengine_amd import _abi, lib
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu

CASES = [
    # n, ic, ih, iw, oc, f, pad, stride
    (1, 32, 1, 1, 32, 1, 0, 1),
    (1, 64, 3, 3, 96, 1, 0, 1),      # nine pixels: the third group of four lanes ends after one
    (3, 32, 5, 7, 160, 3, 1, 1),     # images of 35 pixels, a channel tile that is not full
    (2, 128, 13, 11, 64, 1, 0, 2),
    (1, 64, 18, 15, 32, 3, 1, 1),    # more than one tile of pixels, 270 of them
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_int32_sums(oracle, i):
    n, ic, ih, iw, oc, f, pad, stride = CASES[i]
    kw = dict(pad=pad, stride=stride, dst_dtype=_abi.DT_QS32, scale_bias=1e-4, scale_dst=1e-4)
    d0 = _abi.make_conv_desc("NCHW32", n, ic, ih, iw, oc, f, **kw)
    _, _, _, ds = _abi.conv_shapes(d0)
    d1 = _abi.make_conv_desc("NCHW32", n, ic, ih, iw, oc, f, dst_stride_n=ds[1] * ds[2] * ds[3] * ds[4] + 32, **kw)
    for d in (d0, d1):
        for t in [k for k, name in enumerate(lib.tile_names()) if name in ("v2_128x128x64r4", "v2_64x128x128r3")]:
            assert check_case(oracle, d, seed=90 + i, algo=1, tile=t, tag=lib.tile_names()[t]) is not None
