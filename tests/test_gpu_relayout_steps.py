"""How NCHW <-> NCHW4 conversions are cut into threads: which kernel an exec launches on either side of each line between them (no GPU, for a
device of 256 CUs), and their bytes there.  Images whose last workgroup would be nearly empty must not take the forms that make it
larger."""
import pytest

from megengine_amd import _abi, ops
from tests import routes

ONE, FOUR = "nchw_to_nchw4_kernel<1>", "nchw_to_nchw4_kernel<4>"
P4, P16 = "nchw4_to_nchw_kernel", "nchw4_to_nchw16_kernel"
# images, blocks of four channels, rows, columns; the kernel into NCHW4, the kernel back
LINES = [
    (4096, 1, 32, 32, ONE, P4),          # 2^20 steps, 256 to an image: a quarter of the lanes of four steps
    (2873, 2, 26, 28, ONE, P16),         # 364 steps to an image: a third of them; one workgroup of 16 pixels
    (1500, 1, 37, 76, ONE, P16),         # 703 to an image
    (1500, 1, 44, 64, FOUR, P16),        # 704
    (1024, 1, 64, 65, ONE, P4),          # 1040: two workgroups, 0.51 of their lanes; of 16 pixels 260, also two
    (600, 1, 64, 112, FOUR, P16),        # 1792: 0.88; 448 of 16 pixels
    (600, 1, 65, 110, ONE, P4),          # 1788; 447
    (255, 1, 128, 128, ONE, P16),        # 4096 to an image, just short of 2^20 steps
    (256, 1, 128, 128, FOUR, P16),
    (2047, 1, 128, 128, FOUR, P16),      # just short of 2^23
    (2048, 1, 128, 128, ONE, P16),
    (511, 1, 16, 64, ONE, P4),           # 256 to an image: as many workgroups either way
    (511, 1, 13, 79, ONE, P16),          # 257: one against two
    (300, 1, 30, 46, ONE, P4),           # 345 to an image, too few of them in all
    (63, 1, 128, 128, ONE, P4),          # just short of 2^18
    (64, 1, 128, 128, ONE, P16),
    (64, 16, 56, 56, ONE, P16),
    (3, 1, 224, 224, ONE, P4),
]


def _descs(n, blocks, h, w):
    return (ops.relayout_desc(_abi.RL_NCHW_NCHW4, (n, blocks * 4, h, w)), ops.relayout_desc(_abi.RL_NCHW4_NCHW, (n, blocks, h, w, 4)))


def test_route():
    got = routes.routes([d for line in LINES for d in _descs(*line[:4])])
    for i, line in enumerate(LINES):
        assert [k for r in got[2 * i:2 * i + 2] for k in r.kernels] == list(line[4:]), line


@pytest.mark.gpu
@pytest.mark.parametrize("n,blocks,h,w", [line[:4] for line in LINES if line[0] * line[1] * line[2] * line[3] < 2 ** 24])
def test_bytes(n, blocks, h, w):
    """A conversion moves bytes, so torch's own copies are the reference."""
    import torch
    x = torch.randint(-128, 128, (n, blocks, 4, h, w), dtype=torch.int8, device="cuda")
    to, back = _descs(n, blocks, h, w)
    y = ops.relayout_exec(to, x.view(n, blocks * 4, h, w))
    assert torch.equal(y, x.permute(0, 1, 3, 4, 2))
    assert torch.equal(ops.relayout_exec(back, y).view_as(x), x)
