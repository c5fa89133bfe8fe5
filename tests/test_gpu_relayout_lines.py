"""NCHW -> NCHW32 with stores of whole lines or of half pixels: which of the two an exec launches on either side of the line between them (no GPU,
for a device of 256 CUs), and its bytes there, in tiles that end inside a wave's pixels, inside a group of four and with channels missing."""
import pytest

from megengine_amd import _abi, ops
from tests import routes

LINES = [
    # images, channels, rows, columns; whole lines
    (64, 128, 16, 32, False), (128, 128, 16, 32, True), (127, 128, 16, 32, False),     # two workgroups to a CU
    (128, 100, 12, 32, True), (128, 100, 11, 33, False),                               # three quarters of a tile
    (256, 128, 16, 16, True), (256, 128, 15, 17, False), (255, 128, 16, 16, False),    # four to a CU, half a tile
    (60, 161, 23, 47, True),                                                           # 1081 pixels: the last tile of three holds 57
    (257, 33, 61, 9, True), (171, 75, 13, 60, True), (7, 70, 31, 33, False),
]


def test_route():
    got = routes.routes([ops.relayout_desc(_abi.RL_NCHW_NCHW32, line[:4]) for line in LINES])
    assert [r.kernels for r in got] == [("nchw_to_nchw32_kernel<%s>" % str(line[4]).lower(),) for line in LINES]


@pytest.mark.gpu
@pytest.mark.parametrize("n,c,h,w", [line[:4] for line in LINES])
def test_bytes(n, c, h, w):
    """A conversion moves bytes, so torch's own copies are the reference."""
    import torch
    x = torch.randint(-128, 128, (n, c, h, w), dtype=torch.int8, device="cuda")
    want = torch.zeros((n, (c + 31) // 32 * 32, h, w), dtype=torch.int8, device="cuda")
    want[:, :c] = x
    y = ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW_NCHW32, (n, c, h, w)), x)
    assert torch.equal(y, want.view(n, -1, 32, h, w).permute(0, 1, 3, 4, 2))
