"""Plain NCHW through packed inputs and the planar epilogue at its edges: channel counts on both sides of the packing switch,
planes around the 64 and 128 pixels of a conversion tile, output planes that are no multiple of 4 (groups of four pixels
that straddle two images), odd channel counts, group boundaries inside a channel tile, misaligned tensors.  Most square filters run
in one launch without packing (test_gpu_nchw_patch.py); the sizes that do are here again with filters that are packed."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, lib, ops
from tests import util
from tests.gpu_util import check_case
from tests.routes import routes

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
NCHW = 4
CASES = [
    # n, ic, ih, iw, oc, f, pad, stride, group
    (1, 1, 1, 1, 1, 1, 0, 1, 1),
    (3, 3, 9, 7, 5, 3, 1, 1, 1),
    (2, 16, 8, 8, 33, 3, 1, 1, 1),
    (2, 17, 7, 9, 31, 3, 1, 2, 1),        # 63 input pixels: quads, not tiles
    (3, 40, 8, 8, 96, 1, 0, 1, 1),        # 64
    (2, 33, 127, 1, 130, (3, 1), (1, 0), 1, 1),
    (5, 65, 3, 43, 70, 3, 1, 1, 1),       # 129
    (40, 48, 13, 13, 66, 3, 1, 1, 1),     # enough pixels for the tiled kernel, 169 per image
    (6, 40, 57, 45, 140, 3, 1, 1, 1),
    (2, 192, 9, 9, 128, 3, 1, 1, 2),
    (3, 64, 11, 11, 192, 5, 2, 1, 2),     # 96 channels per group: a tile of 64 ends inside one
    (3, 3, 9, 7, 5, (3, 2), 1, 1, 1),
    (2, 16, 8, 8, 33, (3, 2), (1, 0), 1, 1),
    (2, 17, 7, 9, 31, (2, 3), 1, 2, 1),
    (3, 40, 8, 8, 96, (1, 2), 0, 1, 1),
    (40, 48, 13, 13, 66, (3, 1), (1, 0), 1, 1),
    (6, 40, 57, 45, 140, (1, 3), (0, 1), 1, 1),
]
ONE_LAUNCH = (1, 2, 3, 4, 7, 8)


@pytest.mark.parametrize("i", range(len(CASES)))
def test_edges(oracle, i):
    n, ic, ih, iw, oc, f, pad, stride, group = CASES[i]
    fh, fw = f if isinstance(f, tuple) else (f, f)
    for nl, kw in (("RELU", dict(has_z=True)), ("IDENTITY", dict()), ("H_SWISH", dict(has_z=True, bias_mode=_abi.BIAS_NONE))):
        d = _abi.make_conv_desc("NCHW", n, ic, ih, iw, oc, fh, fw, pad=pad, stride=stride, group=group, nonline=nl, **kw, **S)
        assert (routes([(d, NCHW, -1, True)])[0].kernels[0] == "nchw_prep_kernel") == (i not in ONE_LAUNCH)
        check_case(oracle, d, seed=30 + i, algo=NCHW, tag="nchw planar %d" % i)


@pytest.mark.parametrize("fh,fw", [(3, 6), (2, 9), (18, 1), (1, 9)])
@pytest.mark.parametrize("n,ic,oc", [(2, 12, 45), (2, 75, 70), (24, 40, 66)])   # packed by 4, by 32; pixels for the tiled kernel
def test_filters_that_are_not_square(oracle, n, ic, oc, fh, fw):
    d = _abi.make_conv_desc("NCHW", n, ic, 21, 23, oc, fh, fw, pad=(fh // 2, fw // 2), stride=(1, 2), nonline="RELU", has_z=True, **S)
    assert routes([(d, NCHW, -1, True)])[0].kernels[0] == "nchw_prep_kernel"
    check_case(oracle, d, seed=fh * fw + n, algo=NCHW, tag="nchw planar %dx%d" % (fh, fw))


def test_tensors_at_any_address(oracle):
    d = _abi.make_conv_desc("NCHW", 3, 37, 19, 21, 45, 3, pad=1, nonline="RELU", has_z=True, **S)
    src, flt, bias, z = util.make_tensors(d, seed=9)
    want = oracle.conv_bias(d, src, flt, bias, z)
    algo, ws = ops.conv_bias_query(d, NCHW)
    for off in (1, 2, 3):
        def shifted(x):
            buf = torch.empty(x.size + 16, dtype=torch.int8, device="cuda")
            view = buf[off:off + x.size]
            view.copy_(torch.from_numpy(x.reshape(-1)).cuda())
            return view
        dst = torch.full((want.size + 16,), 77, dtype=torch.int8, device="cuda")
        out = dst[off:off + want.size]
        ops.conv_bias_exec(d, shifted(src), shifted(flt), torch.from_numpy(bias).cuda(), shifted(z), out, algo,
                           torch.empty(ws, dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want.reshape(-1))
        assert int((dst[:off] != 77).sum()) == 0 and int((dst[off + want.size:] != 77).sum()) == 0
