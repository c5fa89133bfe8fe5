"""NCHW <-> NCHW32 where a plane ends inside sixteen bytes, every number of them: the load that ends with the plane and is turned to the front, the
store in eights, fours, twos and ones (relayout_parts.h); in the first plane of the tensor and the last, whose neighbours are not the tensor's; with an
incomplete block of channels; and through the preparation pass of plain NCHW convolutions."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tail", range(16))
@pytest.mark.parametrize("base,c", [(128, 32), (512, 45), (624, 3)])
def test_plane_tails(tail, base, c):
    hw = base + tail
    rng = np.random.RandomState(tail)
    x = rng.randint(-128, 128, (2, c, 1, hw)).astype(np.int8)
    cb = (c + 31) // 32
    padded = np.zeros((2, cb * 32, hw), np.int8)
    padded[:, :c] = x.reshape(2, c, hw)
    want = padded.reshape(2, cb, 32, hw).transpose(0, 1, 3, 2).reshape(2, cb, 1, hw, 32)

    def guarded(shape):   # between guard bytes, which no store may touch
        t = torch.full((int(np.prod(shape)) + 64,), 77, dtype=torch.int8, device="cuda")
        return t, t[32:-32].view(shape)

    src = torch.from_numpy(x).cuda()
    all_y, y = guarded(want.shape)
    ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW_NCHW32, x.shape), src, y)
    assert np.array_equal(y.cpu().numpy(), want)
    if c % 32 == 0:
        all_z, z = guarded(x.shape)
        ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW32_NCHW, want.shape), y, z)
        assert np.array_equal(z.cpu().numpy(), x)
        assert (all_z[:32] == 77).all() and (all_z[-32:] == 77).all()
    assert (all_y[:32] == 77).all() and (all_y[-32:] == 77).all()


@pytest.mark.parametrize("w", range(65, 81))
def test_packed_plain_convolution(oracle, w):
    """one row of 65 to 80 pixels, a filter that only the packed kernels take"""
    d = _abi.make_conv_desc("NCHW", 2, 40, 1, w, 64, 1, 7, pad=(0, 3), nonline="RELU", scale_bias=2e-4, scale_dst=0.05)
    check_case(oracle, d, seed=w, algo=lib.algo_names().index("MI355_NCHW_RELAYOUT_MFMA_I8"), tag="tail %d" % w)
