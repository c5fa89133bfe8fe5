"""Plain NCHW in one launch on tiles that are runs of pixels in the order of memory (conv_patch1.hip): runs that begin and end inside a row,
images whose last group of four is incomplete, several images in a tile, a last run that is nearly empty, one-pixel-wide images out, strides,
and sizes on either side of the rule, which the tile's LDS tells apart.  Against the oracle, and over the residual."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, ops
from tests import util
from tests.routes import UNNAMED, routes

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
CASES = [
    # n, ic, ih, iw, oc, f, pad, stride, bytes of the tile's LDS
    # runs
    (1, 11, 8, 15, 9, 3, 1, 1, 31808),       # 120 pixels, one run of an image
    (3, 17, 45, 13, 33, 3, 1, 1, 35648),     # runs of 120: they begin inside rows
    (8, 6, 92, 11, 126, 3, 1, 1, 34368),
    (2, 9, 25, 41, 70, 5, 2, 2, 50496),      # stride 2
    (14, 15, 74, 59, 34, 5, 2, 1, 49216),    # tiles of 256 pixels
    (9, 20, 4, 4, 33, 3, 0, 3, 68160),       # one pixel out, 32 images in a tile
    (23, 5, 7, 5, 40, 3, 1, 1, 39744),       # images of 35 pixels, three in a tile, the last tile with two
    (701, 5, 7, 9, 40, 3, 0, 1, 56640),      # seven in a tile of 256
    # rows and columns: a run's patch would be more than ...
    (11, 5, 7, 9, 40, 3, 1, 1, 30528),       # 1.3 times as large where every tile has a CU,
    (6, 51, 95, 51, 30, 1, 0, 1, 18560),     # 1.6 times as large in all,
    (38, 13, 42, 21, 172, 1, 0, 1, 40576),   # one quad a thread
    (2, 6, 44, 44, 30, 3, 1, 1, 33344),      # rows of whole groups
]


def desc(c, nl, z, **kw):
    n, ic, ih, iw, oc, f, pad, stride, _ = c
    return _abi.make_conv_desc("NCHW", n, ic, ih, iw, oc, f, pad=pad, stride=stride, nonline=nl, has_z=z, **dict(S, **kw))


def test_rule():
    got = routes([(desc(c, "RELU", True), UNNAMED, -1, False) for c in CASES])
    assert [g.lds for g in got] == [c[-1] for c in CASES]
    assert all(g.kernels[0].startswith("patch1_kernel") for g in got)


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_runs(oracle, i):
    for nl, has_z in (("RELU", True), ("IDENTITY", False), ("H_SWISH", True)):
        d = desc(CASES[i], nl, has_z)
        src, flt, bias, z = util.make_tensors(d, seed=300 + i)
        want = oracle.conv_bias(d, src, flt, bias, z)
        dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]
        assert np.array_equal(ops.conv_bias_exec(d, *dev).cpu().numpy(), want), (CASES[i], nl)
        if has_z:   # the output over its residual
            assert np.array_equal(ops.conv_bias_exec(d, *dev, dev[3]).cpu().numpy(), want), (CASES[i], nl)
