"""Pointwise NCHW4 layers at stride 1 with four pixels per lane (tiles pw4_stream and pw4_split) where they can go wrong: planes that are no
multiple of four pixels, fewer pixels than a group, several images in one tile, channels around the edges of the 16- and
32-channel blocks and of the waves' shares, reductions that end inside a step or have fewer steps than waves, residuals written in
place, batch strides larger than an image."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, lib, ops
from tests import util
from tests.gpu_util import check_case, to_dev

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
IGEMM = 1
CASES = [
    # n, ic, ih, iw, oc
    (1, 4, 1, 1, 4),          # one pixel, one channel block
    (1, 4, 1, 3, 8),
    (5, 16, 7, 7, 96),        # 49 pixels: the last group of an image holds one
    (3, 24, 5, 6, 144),       # 30 pixels: two
    (7, 36, 3, 5, 100),       # 15 pixels: three; two k-steps, the second of one block
    (2, 64, 33, 31, 68),
    (1, 16, 56, 56, 1024),    # the most channels of the streaming kernel
    (2, 64, 9, 8, 1100),
    (40, 32, 28, 28, 192),    # several blocks per wave
    (2, 68, 5, 5, 32),        # just past 64 bytes
    (3, 144, 9, 7, 20),
    (2, 192, 7, 7, 36),
    (1, 960, 7, 7, 160),
    (9, 576, 6, 6, 96),
    (1, 2052, 3, 3, 52),      # 33 steps, the last of one block
    (64, 384, 14, 14, 64),
]


def _tiles():
    return [t for t, name in enumerate(lib.tile_names()) if name in ("pw4_stream", "pw4_split")]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_edges(oracle, i):
    n, ic, ih, iw, oc = CASES[i]
    for nl, z in (("RELU", True), ("IDENTITY", False), ("RELU", False), ("H_SWISH", True)):
        d = _abi.make_conv_desc("NCHW4", n, ic, ih, iw, oc, 1, nonline=nl, has_z=z, **S)
        ran = [check_case(oracle, d, seed=120 + i, algo=IGEMM, tile=t, tag=lib.tile_names()[t]) is not None for t in _tiles()]
        assert ran[1] and (ran[0] or ic > 64 or oc > 1024)


@pytest.mark.parametrize("ic", (24, 144))
def test_strided_batches_and_residual_in_place(oracle, ic):
    d = _abi.make_conv_desc("NCHW4", 3, ic, 5, 7, 40, 1, nonline="RELU", has_z=True, **S)
    d.src_stride_n, d.z_stride_n, d.dst_stride_n = ic * 35 + 20, 40 * 35 + 4, 40 * 35 + 12
    for t in _tiles():
        check_case(oracle, d, seed=140, algo=IGEMM, tile=t, tag=lib.tile_names()[t])
    d = _abi.make_conv_desc("NCHW4", 3, ic, 5, 7, 40, 1, nonline="RELU", has_z=True, **S)
    src, flt, bias, z = util.make_tensors(d, seed=141)
    a, _ = ops.conv_bias_query(d, IGEMM)
    assert a.tile_cfg in _tiles()
    zd = to_dev(z)
    ops.conv_bias_exec(d, to_dev(src), to_dev(flt), to_dev(bias), zd, zd, a)
    torch.cuda.synchronize()
    assert np.array_equal(zd.cpu().numpy(), oracle.conv_bias(d, src, flt, bias, z))
