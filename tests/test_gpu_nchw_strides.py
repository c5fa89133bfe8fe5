"""Plain NCHW layers at stride 2 on both sides of the lines where the one-launch kernel gives way to the packed path (three and four channel
tiles, workgroups per CU, residual, rows out that are not whole quads, rounds of long chains), and 5x5 layers on both sides of its
price: the heuristic's result is the generic kernel's."""
import pytest
import torch

from megengine_amd import _abi, ops
from tests.routes import routes

pytestmark = pytest.mark.gpu

DIRECT = 0


@pytest.mark.parametrize("n,ic,h,w,oc,f,stride,z,packed", [
    (40, 5, 75, 49, 185, 3, 2, False, True),     # three tiles, few channels in
    (26, 35, 95, 75, 161, 1, 2, False, True),    # channels in over a block of 32
    (26, 35, 95, 75, 161, 1, 2, True, False),    # the same with a residual
    (40, 5, 75, 49, 128, 3, 2, False, False),    # two channel tiles
    (24, 3, 91, 96, 150, 3, 2, False, False),    # rows out of whole quads
    (18, 5, 75, 49, 185, 3, 2, False, False),    # fewer workgroups
    (40, 5, 75, 49, 197, 3, 2, True, True),      # four tiles
    (40, 5, 75, 49, 197, 1, 2, True, False),
    (33, 101, 65, 108, 243, 1, 2, False, True),
    (20, 219, 106, 28, 207, 1, 2, False, True),  # another round of four stages
    (21, 234, 51, 33, 191, 3, 2, False, True),
    (24, 182, 28, 11, 52, 5, 1, False, True),    # 5x5
    (11, 47, 34, 51, 252, 5, 2, True, False),
    (30, 193, 12, 18, 169, 5, 2, False, True),
    (12, 25, 14, 87, 132, 5, 1, True, False),
])
def test_both_ways(n, ic, h, w, oc, f, stride, z, packed):
    d = _abi.make_conv_desc("NCHW", n, ic, h, w, oc, f, pad=f // 2, stride=stride, nonline="RELU", has_z=z, scale_bias=2e-4, scale_z=0.05,
                            scale_dst=0.05)
    src_s, flt_s, bias_s, dst_s = _abi.conv_shapes(d)
    g = torch.Generator(device="cuda")
    g.manual_seed(n + oc)
    s8 = lambda shape: torch.randint(-128, 128, shape, generator=g, device="cuda", dtype=torch.int8)  # noqa: E731
    src, flt, zt = s8(src_s), s8(flt_s), s8(dst_s) if z else None
    bias = torch.randint(-4000, 4000, bias_s, generator=g, device="cuda", dtype=torch.int32)
    a, _ = ops.conv_bias_query(d)
    assert a.id != DIRECT and (routes([d])[0].kernels[0] == "nchw_prep_kernel") == packed
    b, _ = ops.conv_bias_query(d, DIRECT)
    got, want = ops.conv_bias_exec(d, src, flt, bias, zt), ops.conv_bias_exec(d, src, flt, bias, zt, None, b)
    assert int((want != 0).sum()) > want.numel() // 8
    assert torch.equal(got, want)
