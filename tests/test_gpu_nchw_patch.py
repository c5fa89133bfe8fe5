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
from tests.routes import UNNAMED, routes

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
CASES = [
    # n, ic, ih, iw, oc, f, pad, stride, tile (blocks of 32 channels, of 128 pixels)
    (1, 5, 1, 4, 1, 1, 0, 1, (1, 1)),            # one row of one quad
    (3, 3, 5, 5, 2, 3, 1, 1, (1, 1)),            # six rows of filter: the last quad passes the filter's end
    (1, 1, 4, 5, 4, 3, 1, 1, (1, 1)),            # four one-channel rows, every quad past the end but the first
    (2, 16, 7, 6, 33, 3, 1, 1, (1, 1)),          # one group, a channel past a tile, several images in a tile
    (3, 17, 9, 11, 31, 3, 0, 2, (1, 1)),         # a group of one channel
    (2, 33, 13, 13, 64, 5, 2, 1, (1, 1)),        # 25 taps: an odd number of entries
    (2, 37, 12, 10, 40, 5, 4, 2, (1, 1)),        # padding of a whole filter: quads entirely outside
    (1, 65, 6, 131, 70, 3, 1, 1, (1, 1)),        # rows wider than a tile
    (5, 64, 3, 43, 66, 1, 0, 1, (1, 1)),
    (2, 130, 8, 9, 35, 1, 0, 2, (1, 1)),
    (2, 20, 18, 19, 24, 3, 2, 3, (1, 1)),        # stride 3
    (12, 18, 63, 61, 40, 3, 1, 1, (1, 2)),
    (24, 9, 62, 59, 190, 3, 1, 1, (2, 2)),
    (20, 21, 65, 63, 70, 3, 1, 2, (2, 1)),
    (30, 6, 62, 61, 20, 5, 2, 1, (1, 2)),
    (9, 150, 5, 5, 12, 3, 1, 1, (1, 1)),         # few tiles, a long reduction: packed by the algorithm of that name
    (12, 7, 61, 73, 30, 1, 0, 1, (1, 2)),    # every tile with every filter
    (14, 9, 57, 59, 190, 1, 0, 1, (2, 2)),
    (14, 13, 71, 73, 70, 1, 0, 2, (2, 1)),
    (14, 3, 57, 59, 190, 5, 2, 1, (2, 2)),
    (12, 5, 67, 65, 70, 5, 2, 2, (2, 1)),
    (2, 1, 6, 5, 5, 5, 2, 1, (1, 1)),        # filters that end inside the quads of their last three rows, and of the last row alone
    (1, 2, 5, 7, 2, 3, 1, 1, (1, 1)),
    (1, 3, 6, 9, 33, 5, 2, 2, (1, 1)),
    (1, 18, 9, 9, 65, 3, 1, 1, (1, 1)),
    (1, 35, 9, 9, 34, 1, 0, 1, (1, 1)),
]


def run(d, dev, dst, workspace):
    n = 0 if workspace is None else workspace.numel()
    rc = lib.lib().mi355_convbias_s8_exec(ops._stream(), d, None, *[ops._ptr(t) for t in dev], ops._ptr(dst), ops._ptr(workspace), n)
    assert rc == 0, lib.lib().mi355_last_error()
    torch.cuda.synchronize()
    return dst.cpu().numpy()


@pytest.mark.parametrize("i", range(len(CASES)))
def test_edges(oracle, i):
    n, ic, ih, iw, oc, f, pad, stride, tile = CASES[i]
    for nl, kw in (("RELU", dict(has_z=True)), ("IDENTITY", dict()), ("H_SWISH", dict(has_z=True, bias_mode=_abi.BIAS_NONE))):
        d = _abi.make_conv_desc("NCHW", n, ic, ih, iw, oc, f, pad=pad, stride=stride, nonline=nl, **kw, **S)
        src, flt, bias, z = util.make_tensors(d, seed=60 + i)
        want = oracle.conv_bias(d, src, flt, bias, z)
        dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]
        assert routes([(d, UNNAMED, -1, False)])[0].kernels == ("patch1_kernel<%d, %d, %d>" % (tile + (f * f,)),)
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
    """The generic kernel named by the caller, and scales outside the fast forms, which the planar kernel does not take: the kernels that
    run, and what they compute."""
    for kw, unnamed in ((S, "patch1_kernel<1, 1, 9>"), (dict(scale_bias=2e-4, scale_dst=1e-42), "conv_direct_kernel")):
        d = _abi.make_conv_desc("NCHW", 2, 11, 9, 9, 13, 3, pad=1, nonline="RELU", **kw)
        assert [r.kernels for r in routes([(d, 0, -1, False), (d, UNNAMED, -1, False)])] == [("conv_direct_kernel",), (unnamed,)]
        src, flt, bias, _ = util.make_tensors(d, seed=3)
        want = oracle.conv_bias(d, src, flt, bias, None)
        dev = [torch.from_numpy(x).cuda() for x in (src, flt, bias)] + [None]
        algo, _ = ops.conv_bias_query(d, 0)
        assert np.array_equal(ops.conv_bias_exec(d, *dev, algo=algo).cpu().numpy(), want)
        assert np.array_equal(run(d, dev, torch.empty_like(torch.from_numpy(want)).cuda(), None), want)


PACKED = [
    # on one side of each line the algorithm packs, on the other it does not: n, ic, ih, iw, oc, f, pad, stride, packs
    (9, 150, 5, 5, 12, 3, 1, 1, False),      # several images in a tile; below 2^22 multiply-adds nothing is packed unless named
    (3, 150, 14, 14, 44, 3, 1, 1, True),     # few tiles, a long reduction
    (3, 40, 14, 14, 44, 3, 1, 1, False),     # a short one
    (7, 60, 29, 31, 64, 3, 1, 1, False),     # 64 workgroups
    (3, 60, 29, 31, 64, 3, 1, 1, True),      # fewer, from 2^24 multiply-adds on
    (2, 33, 13, 13, 64, 5, 2, 1, True),
    (1, 65, 6, 131, 70, 3, 1, 1, True),
]


@pytest.mark.parametrize("i", range(len(PACKED)))
def test_both_ways(oracle, i):
    """The heuristic's choice with a workspace, which it writes where it packs and leaves alone where it does not"""
    n, ic, ih, iw, oc, f, pad, stride, packs = PACKED[i]
    for nl, z in (("RELU", True), ("H_SWISH", False)):
        d = _abi.make_conv_desc("NCHW", n, ic, ih, iw, oc, f, pad=pad, stride=stride, nonline=nl, has_z=z, **S)
        assert (routes([(d, UNNAMED, -1, True)])[0].kernels[0] == "nchw_prep_kernel") == packs
        src, flt, bias, zt = util.make_tensors(d, seed=90 + i)
        want = oracle.conv_bias(d, src, flt, bias, zt)
        dev = [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, zt)]
        _, ws = ops.conv_bias_query(d, 4)
        room = torch.full((ws,), 113, dtype=torch.uint8, device="cuda")
        assert np.array_equal(run(d, dev, torch.empty_like(torch.from_numpy(want)).cuda(), room), want)
        assert bool((room != 113).any()) == packs
