"""Long filter rows in the reference layout on the tiles that split the reduction over waves (v2_ks_*): from a line on they are loaded as
whole lines and turned in LDS.  Reductions on both sides of the line, pieces that end inside a stage of 128 bytes, an odd number of 32-byte
chunks, channels and pixels past the tile, both forms of the kernel's argument; every byte against the oracle, and which kernel runs."""
import pytest

from megengine_amd import _abi, lib
from tests import routes
from tests.gpu_util import check_case

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05, nonline="RELU")
# tile, k of the kernel's template, bytes of a row on the line
TILES = [("v2_ks_64x32w8", "32, 2, 8", 3072), ("v2_ks_32x32w8", "32, 1, 8", 3072), ("v2_ks_16x16w4", "16, 1, 4", 2560),
         ("v2_ks_16x16w8", "16, 1, 8", 5120), ("v2_ks_32x32w4", "32, 1, 4", None)]


def _cases(line):
    # n, ic, h, w, oc, f, stride
    line = line or 1536
    yield 1, line - 32, 5, 7, 96, 1, 1              # below the line
    yield 1, line, 5, 7, 96, 1, 1                   # whole stages, a channel tile that is half empty
    yield 2, line + 32, 4, 9, 32, 1, 1              # an odd number of chunks: pieces of different lengths
    yield 1, line + 96, 3, 5, 160, 1, 2             # pieces that end inside a stage
    yield 2, line // 288 // 32 * 32 + 352, 6, 5, 64, 3, 1   # windows over every border
    yield 1, 32 * (line // 800 + 2), 7, 6, 96, 5, 2


@pytest.mark.parametrize("tile,args,line", TILES)
def test_route(tile, args, line):
    t = lib.tile_names().index(tile)
    ds = [_abi.make_conv_desc("NCHW32", n, ic, h, w, oc, f, pad=f // 2, stride=s, **S) for n, ic, h, w, oc, f, s in _cases(line)]
    for d, got in zip(ds, routes.routes([(d, 1, t, False) for d in ds])):
        k = d.ic * d.fh * d.fw
        name = "ks_turn_kernel<32, %s" if line and k >= line and not (args == "32, 2, 8" and d.oc <= 32) else "ks_kernel<32, %s"
        assert name % args in got.kernels[-1], (k, got.kernels)


@pytest.mark.gpu
@pytest.mark.parametrize("tile,args,line", TILES)
def test_filter_rows(oracle, tile, args, line):
    t = lib.tile_names().index(tile)
    for i, (n, ic, h, w, oc, f, s) in enumerate(_cases(line)):
        for gap in (False, True):   # gaps between the images: the wide argument
            d = _abi.make_conv_desc("NCHW32", n, ic, h, w, oc, f, pad=f // 2, stride=s, has_z=i % 2 == 1, **S)
            if gap:
                d.src_stride_n = ic * h * w + 128
            assert check_case(oracle, d, seed=70 + i, algo=1, tile=t, tag="%s %d" % (tile, i)) is not None
