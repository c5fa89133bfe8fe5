"""Windowed layers whose stages two groups of waves share (conv_patch4.hip, conv_patch1.hip, tiles of 32 x 128): odd and even numbers of stages, an
incomplete last one, either side of the number of workgroups where it begins, every requantisation form of either half of a block with and without
a residual.  Against the oracle; which form runs, by the workgroup's threads."""
import itertools

import numpy as np
import pytest
import torch

from megengine_amd import _abi, lib, ops
from tests import util
from tests.routes import UNNAMED, routes

SCALES = [
    dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05),       # the quotient form
    dict(scale_bias=1.3e-3, scale_z=0.05, scale_dst=0.0271),   # a linear form for IDENTITY and RELU without a residual
]
IGEMM = 1
CASES = [
    # format, n, ic, ih, iw, oc, f, pad, stride, threads of a workgroup
    ("NCHW4", 2, 72, 11, 13, 36, 3, 1, 1, 512),      # three stages, the last one with one group of channels
    ("NCHW4", 1, 132, 9, 30, 20, 3, 1, 1, 512),      # five stages, 20 of 32 channels
    ("NCHW4", 3, 36, 12, 17, 44, 5, 2, 1, 512),      # three stages of 25 taps
    ("NCHW4", 5, 68, 15, 15, 64, 3, 1, 2, 512),
    ("NCHW4", 2, 40, 10, 10, 24, (2, 2), 0, 1, 512),  # two stages
    ("NCHW4", 8, 96, 32, 32, 128, 3, 1, 1, 512),     # 32 workgroups to an XCD
    ("NCHW4", 9, 96, 32, 32, 128, 3, 1, 1, 256),     # 36
    ("NCHW4", 2, 64, 11, 13, 36, 5, 2, 1, 512),
    ("NCHW4", 1, 52, 14, 40, 24, (1, 25), (0, 12), 1, 512),   # 25 taps in a row
    ("NCHW4", 40, 20, 21, 22, 40, 5, 2, 1, 256),     # 25 taps, one group of waves
    ("NCHW", 1, 75, 13, 11, 35, 3, 1, 1, 512),       # three stages, the last one with eleven channels
    ("NCHW", 1, 130, 16, 17, 20, 1, 0, 1, 512),      # three stages of 64
    ("NCHW", 1, 33, 12, 19, 70, 5, 2, 2, 512),
    ("NCHW", 1, 150, 15, 14, 20, 3, 1, 2, 512),
    ("NCHW", 3, 40, 9, 7, 33, 3, 1, 1, 256),         # two stages
    ("NCHW", 64, 75, 16, 16, 33, 3, 1, 1, 512),      # 32 workgroups to an XCD
    ("NCHW", 65, 75, 16, 16, 33, 3, 1, 1, 256),      # 34
    ("NCHW", 64, 130, 16, 16, 33, 1, 0, 1, 512),
    ("NCHW", 65, 130, 16, 16, 33, 1, 0, 1, 256),
]


def _desc(c, nl, z, scales=SCALES[0]):
    fmt, n, ic, ih, iw, oc, f, pad, stride, _ = c
    f = f if isinstance(f, tuple) else (f, f)
    return _abi.make_conv_desc(fmt, n, ic, ih, iw, oc, *f, pad=pad, stride=stride, nonline=nl, has_z=z, **scales)


def _exec(c, d):
    """how the case is run: the tile by name, or (plain NCHW) without an algorithm or a workspace"""
    return (d, IGEMM, lib.tile_names().index("patch4_32x128"), False) if c[0] == "NCHW4" else (d, UNNAMED, -1, False)


def test_which_form():
    got = routes([_exec(c, _desc(c, "RELU", True)) for c in CASES])
    assert [(r.kernels[0].split("<")[0], r.threads) for r in got] == [("patch4_kernel" if c[0] == "NCHW4" else "patch1_kernel", c[-1]) for c in CASES]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_split(oracle, i):
    c = CASES[i]
    for scales, nl, has_z in itertools.product(SCALES, ("IDENTITY", "RELU", "H_SWISH"), (False, True)):
        d = _desc(c, nl, has_z, scales)
        src, flt, bias, z = util.make_tensors(d, seed=500 + i)
        want = oracle.conv_bias(d, src, flt, bias, z)
        dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]
        _, algo, tile, _ = _exec(c, d)
        a = None
        if c[0] == "NCHW4":
            a = ops.conv_bias_query(d, algo)[0]
            a.tile_cfg = tile
        assert np.array_equal(ops.conv_bias_exec(d, *dev, algo=a).cpu().numpy(), want), (c, nl, has_z, scales)
        if has_z:   # the output over its residual
            assert np.array_equal(ops.conv_bias_exec(d, *dev, dev[3], algo=a).cpu().numpy(), want), (c, nl, has_z, scales)
