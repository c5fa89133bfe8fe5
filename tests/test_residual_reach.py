"""Plain NCHW in one launch and grouped layers on the matrix cores: no lane of a residual load or a store leads out of its tensor, by the kernels'
own offsets (tests/host/reach.cpp, no GPU).  Plain: channels that eight and 32 do not divide, in the last image above all; every tile; runs and
rows that end inside a group of four; planes that hold no dword; images apart.  Grouped: planes of fewer pixels than a step, bands."""
import os
import subprocess

import pytest

from megengine_amd import _abi

HERE = os.path.dirname(os.path.abspath(__file__))
EXE = os.path.join(HERE, "host", "reach")

CASES = [
    # n, ic, ih, iw, oc, f, pad, stride; blocks of 32 channels and of 128 pixels of the tile
    (6, 75, 61, 45, 150, 3, 1, 1, (1, 2)),
    (1, 8, 9, 9, 1, 5, 0, 1, (1, 1)),
    (2, 5, 8, 11, 33, 3, 1, 1, (1, 1)),
    (3, 40, 20, 17, 70, 5, 2, 1, (1, 1)),         # two groups of waves
    (70, 4, 5, 5, 41, 5, 0, 1, (1, 1)),           # planes of one byte
    (7000, 4, 5, 6, 35, 5, 0, 1, (1, 2)),         # of two, on a tile of 256 pixels
    (5000, 4, 3, 8, 69, 3, 0, 5, (2, 1)),         # at a stride
    (16400, 3, 5, 6, 70, 5, 0, 1, (2, 2)),        # on the largest
    (70, 20, 45, 37, 27, 3, 1, 1, (1, 2)),
    (64, 8, 31, 63, 189, 3, 1, 1, (2, 2)),
    (64, 8, 41, 43, 70, 1, 0, 1, (2, 2)),
    (64, 16, 61, 61, 100, 3, 1, 2, (2, 1)),
]
GROUPED = [
    # n, groups, channels of one, ih, iw, pad, stride
    (2, 4, 4, 3, 3, 0, 1), (1, 2, 8, 5, 5, 1, 1), (3, 2, 16, 7, 5, 1, 2), (1, 4, 4, 8, 16, 1, 1), (64, 8, 16, 46, 30, 1, 1), (40, 22, 8, 87, 13, 1, 1),
]


def _desc(c, z, gap):
    n, ic, ih, iw, oc, f, pad, stride, _ = c
    d = _abi.make_conv_desc("NCHW", n, ic, ih, iw, oc, f, pad=pad, stride=stride, nonline="RELU", has_z=z, scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
    if gap:
        out = oc * _abi.out_size(ih, f, 1, stride, pad) * _abi.out_size(iw, f, 1, stride, pad)
        d.dst_stride_n, d.z_stride_n = out + 40, out + 24
    return d


def _grouped(c, z, gap):
    n, g, per, ih, iw, pad, stride = c
    d = _abi.make_conv_desc("NCHW4", n, g * per, ih, iw, g * per, 3, pad=pad, stride=stride, group=g, nonline="RELU", has_z=z, scale_bias=2e-4,
                            scale_z=0.05, scale_dst=0.05)
    if gap:   # the kernel's wide argument
        d.dst_stride_n = g * per * _abi.out_size(ih, 3, 1, stride, pad) * _abi.out_size(iw, 3, 1, stride, pad) + 64
    return d


@pytest.mark.parametrize("gap", [False, True])
@pytest.mark.parametrize("z", [False, True])
def test_no_lane_leads_out(z, gap):
    subprocess.check_call(["make", "-C", os.path.dirname(EXE), "-s", EXE])
    descs = [_desc(c, z, gap) for c in CASES] + [_grouped(c, z, gap) for c in GROUPED]
    lines = "".join(bytes(d).hex() + "\n" for d in descs)
    r = subprocess.run([EXE], input=lines, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    got = [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]
    assert [g[:2] for g in got] == [c[-1] for c in CASES] + [(0, 0)] * len(GROUPED)
    assert all(g[2] > 0 for g in got)
    assert [g[3] for g in got] == [0] * len(descs)
