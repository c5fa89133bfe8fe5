"""The tile for a dense 32-packed layer with its filter in the reference layout, at sizes on both sides of the prices' crossings: a tile that
can run the problem, with the oracle's result."""
import pytest

from megengine_amd import _abi, lib, ops
from tests.gpu_util import check_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ic,h,w,oc,f,stride,z,names", [
    (3, 128, 33, 31, 96, 3, 2, True, None),
    (40, 288, 21, 9, 64, 1, 1, False, None),
    (12, 64, 31, 45, 96, 5, 1, True, None),
    (9, 96, 47, 46, 320, 3, 1, False, {"v2_128x256x64r3w8", "dma128x128x128r2w8"}),   # many tiles: the large ones
    (33, 64, 30, 31, 64, 5, 1, False, {"dma64x128x128w8", "v2_64x128x64r4"}),         # 64 channels: no tile of 128
    (9, 96, 31, 33, 160, 1, 1, False, {"pw32_stream"}),                               # pointwise, at most 96 channels, no residual
    (3, 96, 40, 41, 224, 1, 2, False, None),                                          # the same with fewer outputs
])
def test_plain_pick(oracle, n, ic, h, w, oc, f, stride, z, names):
    d = _abi.make_conv_desc("NCHW32", n, ic, h, w, oc, f, pad=f // 2, stride=stride, nonline="RELU", has_z=z, scale_bias=2e-4, scale_z=0.05,
                            scale_dst=0.05)
    a, ws = ops.conv_bias_query(d)
    assert a.id == 1 and ws == 0
    if names:
        assert lib.tile_names()[a.tile_cfg] in names
    check_case(oracle, d, seed=n, tag=lib.tile_names()[a.tile_cfg])
