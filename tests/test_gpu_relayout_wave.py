"""NCHW <-> NCHW32 in tiles of one wave: on either side of the number of workgroups where it ends (for a device of 256 CUs), planes that end inside a
tile, inside sixteen bytes and exactly, incomplete blocks of channels on the way in."""
import pytest

from megengine_amd import _abi, ops
from tests import routes

CASES = [
    # images, channels, rows, columns; threads of a workgroup in and back
    (1, 32, 8, 16, 64, 64), (2, 64, 27, 22, 64, 64), (3, 75, 31, 17, 64, 64), (5, 96, 1, 129, 64, 64), (1, 40, 64, 63, 64, 64),
    (4, 32 * 32, 16, 32, 64, 64), (129, 32, 16, 16, 64, 256),           # 128 and 129 tiles of 512 pixels
    (6, 32 * 32, 20, 13, 64, 256), (193, 32, 16, 16, 256, 256),         # 192 and 193
]


def _descs(n, c, h, w):
    return ops.relayout_desc(_abi.RL_NCHW_NCHW32, (n, c, h, w)), ops.relayout_desc(_abi.RL_NCHW32_NCHW, (n, (c + 31) // 32, h, w, 32))


def test_route():
    for c in CASES:
        got = routes.routes(list(_descs(*c[:4])))
        assert [r.threads for r in got] == list(c[4:]), c
        assert [r.kernels for r in got] == [("nchw_to_nchw32_kernel<false>",), ("nchw32_to_nchw_kernel",)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,c,h,w", [c[:4] for c in CASES])
def test_bytes(n, c, h, w):
    import torch
    x = torch.randint(-128, 128, (n, c, h, w), dtype=torch.int8, device="cuda")
    padded = torch.zeros((n, (c + 31) // 32 * 32, h, w), dtype=torch.int8, device="cuda")
    padded[:, :c] = x
    to, back = _descs(n, c, h, w)
    y = ops.relayout_exec(to, x)
    assert torch.equal(y, padded.view(n, -1, 32, h, w).permute(0, 1, 3, 4, 2))
    assert torch.equal(ops.relayout_exec(back, y), padded)
