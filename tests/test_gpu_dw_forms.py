"""Channel-wise layers on the matrix cores (conv_dwm.hip): every requantisation form, with and without a residual, on either side of the
number of matrix steps from which the form is chosen inside the loop; the output over its residual.  Against the oracle."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, ops
from tests import util
from tests.routes import routes

CASES = [
    # n, channels, ih, iw, filter, stride; matrix steps of a quad
    (1, 8, 23, 22, (1, 7), 1),    # one
    (2, 12, 30, 41, (5, 5), 1),   # three
    (16, 240, 57, 57, (5, 5), 2), # four
    (1, 8, 33, 45, (6, 6), 1),    # five
]
SCALES = [
    dict(scale_bias=1.3e-3, scale_z=0.05, scale_dst=0.0271),   # a linear form for IDENTITY and RELU without a residual
    dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05),       # none: the quotient form
    dict(scale_bias=1e-20, scale_z=3e-19, scale_dst=1e-18),    # the literal chain
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_every_form(oracle, i):
    n, c, ih, iw, f, s = CASES[i]
    for scales in SCALES:
        for nl in ("IDENTITY", "RELU", "H_SWISH"):
            for has_z in (False, True):
                d = _abi.make_conv_desc("NCHW4", n, c, ih, iw, c, *f, pad=(f[0] // 2, f[1] // 2), stride=s, group=c, nonline=nl, has_z=has_z, **scales)
                src, flt, bias, z = util.make_tensors(d, seed=90 + i)
                want = oracle.conv_bias(d, src, flt, bias, z)
                dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]
                assert np.array_equal(ops.conv_bias_exec(d, *dev).cpu().numpy(), want), (CASES[i], nl, has_z, scales)
                if has_z:
                    assert np.array_equal(ops.conv_bias_exec(d, *dev, dev[3]).cpu().numpy(), want), (CASES[i], nl, scales)


def test_route():
    for n, c, ih, iw, f, s in CASES:
        d = _abi.make_conv_desc("NCHW4", n, c, ih, iw, c, *f, pad=(f[0] // 2, f[1] // 2), stride=s, group=c, nonline="RELU", has_z=True, **SCALES[0])
        assert routes([d])[0].kernels[0].startswith("dwm_kernel"), (f, s)
