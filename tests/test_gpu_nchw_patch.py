"""Plain NCHW in one launch (the planar patch kernel) where it can go wrong: rows that end inside a group of four pixels, planes
narrower than a tile and wider than one, several images in a tile, an incomplete channel quad at the very end of the filter,
channel groups that do not fill a stage, strides, paddings wider than the filter, batch strides, tensors at any address, and
sizes on either side of each line of the choice.  Through the heuristic without a workspace, which reaches the kernel at
every size, and with one, against the oracle; the generic kernel, named, stays itself."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, lib, ops
from tests import util

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
CASES = [
    # n, ic, ih, iw, oc, f, pad, stride
    (1, 5, 1, 4, 1, 1, 0, 1),            # one row of one quad
    (3, 3, 5, 5, 2, 3, 1, 1),            # six rows of filter: the last quad passes the filter's end
    (1, 1, 4, 5, 4, 3, 1, 1),            # four one-channel rows, every quad past the end but the first
    (2, 16, 7, 6, 33, 3, 1, 1),          # one group, a channel past a tile, several images in a tile
    (3, 17, 9, 11, 31, 3, 0, 2),         # a group of one channel
    (2, 33, 13, 13, 64, 5, 2, 1),        # 25 taps: an odd number of entries
    (2, 37, 12, 10, 40, 5, 4, 2),        # padding of a whole filter: quads entirely outside
    (1, 65, 6, 131, 70, 3, 1, 1),        # rows wider than a tile
    (5, 64, 3, 43, 66, 1, 0, 1),
    (2, 130, 8, 9, 35, 1, 0, 2),
    (2, 20, 18, 19, 24, 3, 2, 3),        # stride 3
    (12, 18, 63, 61, 40, 3, 1, 1),       # 32 x 256
    (24, 9, 62, 59, 190, 3, 1, 1),       # 64 x 256
    (20, 21, 65, 63, 70, 3, 1, 2),       # 64 x 128
    (30, 6, 62, 61, 20, 5, 2, 1),
    (9, 150, 5, 5, 12, 3, 1, 1),         # few tiles, a long reduction: packed when there is a workspace
]


def run(d, dev, dst, workspace):
    n = 0 if workspace is None else workspace.numel()
    rc = lib.lib().mi355_convbias_s8_exec(ops._stream(), d, None, *[ops._ptr(t) for t in dev], ops._ptr(dst), ops._ptr(workspace), n)
    assert rc == 0, lib.lib().mi355_last_error()
    torch.cuda.synchronize()
    return dst.cpu().numpy()


@pytest.mark.parametrize("i", range(len(CASES)))
def test_edges(oracle, i):
    n, ic, ih, iw, oc, f, pad, stride = CASES[i]
    for nl, kw in (("RELU", dict(has_z=True)), ("IDENTITY", dict()), ("H_SWISH", dict(has_z=True, bias_mode=_abi.BIAS_NONE))):
        d = _abi.make_conv_desc("NCHW", n, ic, ih, iw, oc, f, pad=pad, stride=stride, nonline=nl, **kw, **S)
        src, flt, bias, z = util.make_tensors(d, seed=60 + i)
        want = oracle.conv_bias(d, src, flt, bias, z)
        dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]
        _, ws = ops.conv_bias_query(d, 4)
        for room in (None, torch.empty(ws, dtype=torch.uint8, device="cuda")):
            dst = torch.full((want.size + 8,), 77, dtype=torch.int8, device="cuda")
            got = run(d, dev, dst, room)
            assert np.array_equal(got[:want.size], want.reshape(-1)), (CASES[i], nl, room is None)
            assert (got[want.size:] == 77).all()
        if z is not None:   # the output over its residual
            dst = dev[3].clone().reshape(-1)
            assert np.array_equal(run(d, dev[:3] + [dst], dst, None), want.reshape(-1))


@pytest.mark.parametrize("f", [1, 3, 5])
def test_views_and_addresses(oracle, f):
    """Batch strides larger than an image, and every tensor but the bias at an odd address."""
    one = _abi.make_conv_desc("NCHW", 3, 19, 11, 14, 37, f, pad=f // 2, nonline="RELU", has_z=True, **S)
    src, flt, bias, z = util.make_tensors(one, seed=f)
    want = oracle.conv_bias(one, src, flt, bias, z)
    si, di = src[0].size, want[0].size
    d = _abi.make_conv_desc("NCHW", 3, 19, 11, 14, 37, f, pad=f // 2, nonline="RELU", has_z=True, src_stride_n=si + 5, dst_stride_n=di + 3,
                            z_stride_n=di + 7, **S)

    def spread(x, stride):
        buf = torch.full((3 * stride + 16,), 55, dtype=torch.int8, device="cuda")
        for i in range(3):
            buf[1 + i * stride:1 + i * stride + x[i].size] = torch.from_numpy(x[i].reshape(-1)).cuda()
        return buf
    zs = spread(z, di + 7)
    fb = torch.zeros(flt.size + 16, dtype=torch.int8, device="cuda")
    fb[3:3 + flt.size] = torch.from_numpy(flt.reshape(-1)).cuda()
    dst = torch.full((3 * (di + 3) + 16,), 99, dtype=torch.int8, device="cuda")
    dev = [spread(src, si + 5)[1:], fb[3:], torch.from_numpy(bias).cuda(), zs[1:]]
    got = run(d, dev, dst[1:], None)
    for i in range(3):
        at = i * (di + 3)
        assert np.array_equal(got[at:at + di], want[i].reshape(-1))
        assert (got[at + di:at + di + 3] == 99).all()


def test_what_is_named_runs_as_itself(oracle):
    """The generic kernel named by the caller, and scales outside the fast forms, which the planar kernel does not take."""
    for kw in (S, dict(scale_bias=2e-4, scale_dst=1e-42)):
        d = _abi.make_conv_desc("NCHW", 2, 11, 9, 9, 13, 3, pad=1, nonline="RELU", **kw)
        src, flt, bias, _ = util.make_tensors(d, seed=3)
        want = oracle.conv_bias(d, src, flt, bias, None)
        dev = [torch.from_numpy(x).cuda() for x in (src, flt, bias)] + [None]
        algo, _ = ops.conv_bias_query(d, 0)
        assert np.array_equal(ops.conv_bias_exec(d, *dev, algo=algo).cpu().numpy(), want)
        assert np.array_equal(run(d, dev, torch.empty_like(torch.from_numpy(want)).cuda(), None), want)
