"""Grouped 3x3 layers on the matrix cores (grp16_kernel of conv_group4.hip), one band of rows to a workgroup: every requantisation form with
and without a residual, rows that a step of 128 pixels crosses never, once and many times, bands that end inside a step, an incomplete last
band of several steps at strides 1 and 2, outputs of fewer pixels than a wave's units, and the output over its residual.  Against the oracle.  Bands of
several steps need more workgroups than CUs (the price of g16_band_rows), so which bands a case has is held as well."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, ops
from tests import routes, util

CASES = [
    # n, groups, channels of one, ih, iw, pad, stride; bands of an image, steps of a band
    (1, 4, 4, 5, 130, 1, 1, 5, 2),       # a step is less than a row
    (2, 2, 8, 9, 128, 1, 1, 9, 1),       # exactly a row
    (1, 2, 16, 70, 3, 1, 1, 2, 1),       # a step is 42 rows
    (3, 3, 16, 40, 1, 1, 1, 1, 1),       # one column
    (2, 4, 4, 87, 13, 1, 1, 10, 1),      # bands of rows that do not divide the image
    (9, 32, 4, 23, 45, 1, 2, 3, 1),
    (40, 22, 8, 46, 30, 1, 1, 2, 6),     # equal bands, more workgroups than CUs
    (2, 2, 16, 12, 33, 2, 2, 1, 1),
    (11, 16, 8, 41, 29, 1, 1, 2, 5),     # four or five rows end in a step; a last band of one row less
    (22, 16, 4, 5, 128, 1, 1, 2, 3),     # a step is exactly a row, three of them
    (43, 4, 8, 171, 3, 1, 1, 2, 3),      # 42 rows and two columns further on
    (24, 4, 16, 257, 1, 1, 1, 2, 2),     # one column
    (33, 8, 4, 50, 30, 1, 2, 2, 2),      # stride 2: 13 rows of 15, and 12
    (33, 2, 16, 254, 6, 1, 2, 2, 2),     # 64 rows of 3, and 63
    (2, 4, 4, 3, 3, 0, 1, 1, 1),         # one pixel
    (1, 2, 8, 5, 5, 1, 1, 1, 1),         # 25: nothing left for the next step
    (3, 2, 16, 7, 5, 1, 2, 1, 1),
]
SCALES = [
    dict(scale_bias=1.3e-3, scale_z=0.05, scale_dst=0.0271),   # a linear form for IDENTITY and RELU without a residual
    dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05),       # none: the quotient form
    dict(scale_bias=1e-20, scale_z=3e-19, scale_dst=1e-18),    # not even that: the literal chain
]


def _desc(c, nl, z, scales):
    n, g, per, ih, iw, pad, stride = c[:7]
    return _abi.make_conv_desc("NCHW4", n, g * per, ih, iw, g * per, 3, pad=pad, stride=stride, group=g, nonline=nl, has_z=z, **scales)


def test_route():
    got = routes.routes([_desc(c, "RELU", False, SCALES[0]) for c in CASES])
    assert all(r.kernels == ("grp16_kernel<false>",) for r in got)
    for c, r in zip(CASES, got):
        oh, ow = (_abi.out_size(i, 3, 1, c[6], c[5]) for i in c[3:5])
        bands = r.grid // c[0]
        rows = -(-oh // bands)   # bands are equal, so this is the rows of one
        assert (bands, -(-rows * ow // 128)) == c[7:], c


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_every_form(oracle, i):
    for scales in SCALES:
        for nl in ("IDENTITY", "RELU", "H_SWISH"):
            for has_z in (False, True):
                d = _desc(CASES[i], nl, has_z, scales)
                src, flt, bias, z = util.make_tensors(d, seed=70 + i)
                want = oracle.conv_bias(d, src, flt, bias, z)
                dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]
                assert np.array_equal(ops.conv_bias_exec(d, *dev).cpu().numpy(), want), (CASES[i], nl, has_z, scales)
                if has_z:   # the output over its residual
                    assert np.array_equal(ops.conv_bias_exec(d, *dev, dev[3]).cpu().numpy(), want), (CASES[i], nl, scales)
