"""The two forms of a kernel's argument: a wire of at most 112 bytes where the problem's numbers fit it, the launch code's own struct where they
do not (gaps between the images of a batch, sides of 65536, more work items than the wire's divisions are exact for) or where a launch is
large.  Which one an exec launches (no GPU, through tests/host/route.cpp), and every byte of both forms' results."""
import os
import re
import subprocess

import pytest

from megengine_amd import _abi
from tests import routes

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)


def _desc(fmt, n, ic, h, w, oc, f, gap=None, **kw):
    d = _abi.make_conv_desc(fmt, n, ic, h, w, oc, f, pad=f // 2, **kw, **S)
    if gap == "src":
        d.src_stride_n = ic * h * w + 32 * 4
    elif gap == "dst":
        d.dst_stride_n = oc * ((h + 2 * (f // 2) - f) // d.stride_h + 1) * ((w + 2 * (f // 2) - f) // d.stride_w + 1) + 32 * 4
    elif gap == "z":
        d.z_stride_n = oc * ((h + 2 * (f // 2) - f) // d.stride_h + 1) * ((w + 2 * (f // 2) - f) // d.stride_w + 1) + 32 * 4
    return d


# kernel, format, (n, ic, h, w, oc, f) and the rest: edges of tiles and odd sizes, every family that has a wire
CASES = [
    ("ks_kernel<32, 16, 1, 4, true>", "NCHW32", (2, 64, 11, 13, 96, 1), dict(nonline="RELU")),
    ("ks_kernel<32, 16, 1, 4, false>", "NCHW32", (3, 96, 9, 7, 96, 3), dict(nonline="H_SWISH", stride=2)),
    ("ks_kernel<32, 32, 2, 8, false>", "NCHW32", (2, 64, 21, 19, 352, 5), dict()),
    ("ks_kernel<4, 16, 1, 8, false>", "NCHW4", (2, 132, 9, 11, 36, 3), dict(nonline="RELU")),
    ("patch4_one_kernel<1, 1, 1>", "NCHW4", (2, 20, 9, 11, 36, 3), dict()),
    ("dw3x3_kernel<1, 1, 2, true>", "NCHW4", (3, 20, 13, 17, 20, 3), dict(group=20, nonline="H_SWISH")),
    ("dw3x3_kernel<2, 1, 2, true>", "NCHW4", (3, 20, 13, 17, 20, 3), dict(group=20, stride=2)),
    ("dwf_kernel<5, 1, 1>", "NCHW4", (16, 128, 7, 7, 128, 5), dict(group=128)),
    ("dwm_kernel<4, true>", "NCHW4", (3, 24, 21, 23, 24, 5), dict(group=24, stride=2, nonline="RELU")),
    ("grp4_kernel<1, 3, 1>", "NCHW4", (3, 12, 9, 13, 12, 3), dict(group=3)),
    ("grp16_kernel<true>", "NCHW4", (3, 32, 11, 13, 32, 3), dict(group=4, nonline="RELU")),
    ("grp32_kernel<1, 1, 1>", "NCHW32", (3, 96, 9, 14, 96, 3), dict(group=3, nonline="H_SWISH")),
    ("grp32_kernel<2, 1, 1>", "NCHW32", (4, 128, 29, 30, 192, 3), dict(group=2, stride=2)),
    ("pw32s_kernel<2, 2, false>", "NCHW32", (19, 64, 31, 29, 64, 1), dict(nonline="H_SWISH")),
    ("pw4k_kernel<1, 1>", "NCHW4", (3, 20, 9, 13, 28, 1), dict(nonline="RELU")),
    ("pw4q_kernel<1, 1, true>", "NCHW4", (9, 16, 57, 55, 96, 1), dict(nonline="H_SWISH")),
]


def _forms(descs):
    """the type of the last launch's argument for each descriptor"""
    if not os.path.exists(routes.EXE):
        subprocess.check_call(["make", "-C", os.path.dirname(routes.EXE), "-s", routes.EXE])
    lines = "".join("%s -1 -1 1\n" % bytes(d).hex() for d in descs)
    r = subprocess.run([routes.EXE], input=lines, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:]
    return [re.search(r"(\w+)(?:, [^()]*)?\)$", line).group(1) for line in r.stdout.splitlines()]


def test_which_form():
    wires, wides = [], []
    for kernel, fmt, shape, kw in CASES:
        gaps = (None, "src", "dst") if kernel.endswith("false>") and kernel.startswith("pw32s") else (None, "src", "dst", "z")
        descs = [_desc(fmt, *shape, has_z=len(gaps) == 4, gap=gap, **kw) for gap in gaps]
        for r in routes.routes(descs):
            assert r.kernels[-1].replace("_wire", "") == kernel, (kernel, r.kernels)
        if kernel.startswith("patch4"):
            continue
        forms = _forms(descs)
        assert forms[0].endswith("Wire"), (kernel, forms)
        wires.append(kernel)
        assert all(f.endswith("Wide") for f in forms[1:]), (kernel, forms)
        wides.append(kernel)
    assert len(wires) == len(wides) == len(CASES) - 1


def test_numbers_that_do_not_fit():
    def dw(n, c, h, w):
        return _abi.make_conv_desc("NCHW4", n, c, h, w, c, 3, group=c, pad=1, **S)

    assert _forms([dw(1, 4, 1, 65535), dw(1, 4, 1, 65536), dw(1, 4, 65535, 1), dw(1, 4, 65536, 1)]) == ["Dw3Wire", "Dw3Wide"] * 2
    # (such sides of the other families are the generic kernel's, so that gaps between images are what they meet: above)
    wide = [_desc("NCHW32", 1, 64, 1, 65535, 64, 1), _desc("NCHW4", 1, 12, 3, 65535, 12, 3, group=3), _desc("NCHW32", 1, 64, 3, 65535, 64, 3, group=2)]
    assert all(r.kernels == ("conv_direct_kernel",) for r in routes.routes(wide))
    # work items (four columns of four rows here) that the wire's divisions are exact for: fewer than 2^21
    assert _forms([dw(1, 4 * 127, 4 * 128, 4 * 128), dw(1, 4 * 128, 4 * 128, 4 * 128)]) == ["Dw3Wire", "Dw3Wide"]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_both_forms(i):
    from oracle import oracle
    from tests.gpu_util import check_case
    kernel, fmt, shape, kw = CASES[i]
    for gap in (None, "src", "dst", "z"):
        for has_z in (True, False):
            if gap != "z" or has_z:
                check_case(oracle, _desc(fmt, *shape, has_z=has_z, gap=gap, **kw), seed=i + 5, tag="%s gap %s" % (kernel, gap))


# The sizes where opening the wire in every workgroup begins to cost more than the launch gains: kernel, format, the layer on the wire's
# side of the line and the one beyond, options
SIZE_LINES = [
    ("grp4_kernel<1, 3, 1>", "NCHW4", (56, 36, 7, 9, 36, 3), (57, 36, 7, 9, 36, 3), dict(group=9)),                   # 504, 513 workgroups
    ("grp4_kernel<2, 3, 2>", "NCHW4", (85, 24, 56, 56, 24, 3), (86, 24, 56, 56, 24, 3), dict(group=3, stride=2)),     # 510, 516
    ("ks_kernel<32, 32, 1, 4, false>", "NCHW32", (1, 96, 128, 128, 32, 3), (1, 96, 129, 128, 32, 3), dict()),         # 512, 520
    ("pw4k_kernel<4, 1>", "NCHW4", (145, 72, 29, 31, 36, 1), (146, 72, 29, 31, 36, 1), dict()),                       # 2040, 2056
    ("grp32_kernel<2, 1, 1>", "NCHW32", (20, 128, 29, 30, 192, 3), (21, 128, 29, 30, 192, 3), dict(group=2, stride=2)),   # 240, 288
]


def test_which_form_by_the_size_of_a_launch():
    for kernel, fmt, small, large, kw in SIZE_LINES:
        descs = [_desc(fmt, *small, **kw), _desc(fmt, *large, **kw)]
        assert [r.kernels[-1] for r in routes.routes(descs)] == [kernel] * 2
        small, large = _forms(descs)
        assert small.endswith("Wire") and large.endswith("Wide"), (kernel, small, large)


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(SIZE_LINES)))
def test_both_sides_of_a_size(i):
    from oracle import oracle
    from tests.gpu_util import check_case
    kernel, fmt, small, large, kw = SIZE_LINES[i]
    for shape in (small, large):
        for has_z in (True, False):
            check_case(oracle, _desc(fmt, *shape, has_z=has_z, nonline="RELU", **kw), seed=i + 31, tag=kernel)
