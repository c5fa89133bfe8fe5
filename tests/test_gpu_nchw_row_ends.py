"""Plain NCHW in one launch where rows end inside a group of four columns: the residual of such a group is the dword that ends there, from the first
byte of the tensor on, and its outputs are stored as two bytes and one.  Images of one to seven columns, whose first group has fewer than four bytes
before it; planes that hold no dword; one channel and nine; the largest tile.  Against the oracle, and over the residual."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, ops
from tests import util
from tests.routes import UNNAMED, routes

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
# n, ic, oh, ow, oc
CASES = [(1, 4, 2, w, oc) for w in range(1, 8) for oc in (2, 9)] + [(1, 8, 1, 5, 1), (1, 8, 4, 1, 1), (1, 8, 1, 3, 1), (70, 4, 1, 1, 40), (5, 4, 1, 2, 65), (3, 4, 3, 1, 9), (3, 5, 3, 2, 33), (2, 5, 9, 37, 40), (9, 3, 41, 43, 70)]


def _desc(c, nl, has_z):
    n, ic, oh, ow, oc = c
    return _abi.make_conv_desc("NCHW", n, ic, oh + 4, ow + 4, oc, 5, nonline=nl, has_z=has_z, **S)


def test_route():
    got = routes([(_desc(c, "RELU", True), UNNAMED, -1, False) for c in CASES])
    assert all(r.kernels[0].startswith("patch1_kernel") for r in got)


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_row_ends(oracle, i):
    for nl, has_z in (("RELU", True), ("IDENTITY", True), ("IDENTITY", False), ("H_SWISH", True)):
        d = _desc(CASES[i], nl, has_z)
        src, flt, bias, z = util.make_tensors(d, seed=700 + i)
        want = oracle.conv_bias(d, src, flt, bias, z)
        dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]
        assert np.array_equal(ops.conv_bias_exec(d, *dev).cpu().numpy(), want), (CASES[i], nl)
        if has_z:
            assert np.array_equal(ops.conv_bias_exec(d, *dev, dev[3]).cpu().numpy(), want), (CASES[i], nl)
