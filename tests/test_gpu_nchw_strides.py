"""Plain NCHW layers at stride 2 around the line where the one-launch kernel gives way to the packed path (2000 workgroups, more than
128 channels out, 1x1 and 3x3, no residual, rows out that are not whole quads): the heuristic's result is the generic kernel's."""
import pytest
import torch

from megengine_amd import _abi, ops

pytestmark = pytest.mark.gpu

DIRECT = 0


@pytest.mark.parametrize("n,ic,h,w,oc,f,z", [
    (40, 5, 75, 49, 185, 3, False),     # packed, few channels in
    (26, 35, 95, 75, 161, 1, False),    # packed, channels in over a block of 32
    (26, 35, 95, 75, 161, 1, True),     # the same with a residual: one launch
    (40, 5, 75, 49, 128, 3, False),     # two channel tiles: one launch
    (24, 3, 91, 96, 150, 3, False),     # rows out of whole quads: one launch
    (18, 5, 75, 49, 185, 3, False),     # fewer workgroups: one launch
])
def test_strided(n, ic, h, w, oc, f, z):
    d = _abi.make_conv_desc("NCHW", n, ic, h, w, oc, f, pad=f // 2, stride=2, nonline="RELU", has_z=z, scale_bias=2e-4, scale_z=0.05,
                            scale_dst=0.05)
    src_s, flt_s, bias_s, dst_s = _abi.conv_shapes(d)
    g = torch.Generator(device="cuda")
    g.manual_seed(n + oc)
    s8 = lambda shape: torch.randint(-128, 128, shape, generator=g, device="cuda", dtype=torch.int8)  # noqa: E731
    src, flt, zt = s8(src_s), s8(flt_s), s8(dst_s) if z else None
    bias = torch.randint(-4000, 4000, bias_s, generator=g, device="cuda", dtype=torch.int32)
    a, _ = ops.conv_bias_query(d)
    assert a.id != DIRECT
    b, _ = ops.conv_bias_query(d, DIRECT)
    got, want = ops.conv_bias_exec(d, src, flt, bias, zt), ops.conv_bias_exec(d, src, flt, bias, zt, None, b)
    assert int((want != 0).sum()) > want.numel() // 8
    assert torch.equal(got, want)
