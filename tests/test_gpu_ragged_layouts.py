"""Layout conversions and large-window pooling at the edges of their kernels: image sizes around the 16-pixel vectors and
the LDS tile, channel counts that leave blocks incomplete, windows around the sixteen lanes that share one."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, ops
from tests import util
from tests.gpu_util import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(1, 1), (3, 5), (4, 4), (1, 17), (7, 7), (1, 127), (8, 16), (3, 43), (31, 33), (19, 27), (23, 45)])
@pytest.mark.parametrize("c", [1, 3, 4, 31, 33, 64, 75])
def test_plain_to_packed_and_back(oracle, h, w, c):
    x = util.uniform_int(7 * h + w + c, (3, c, h, w), -128, 127, np.int8)
    modes = [(_abi.RL_NCHW_NCHW4, _abi.RL_NCHW4_NCHW), (_abi.RL_NCHW_NCHW32, _abi.RL_NCHW32_NCHW)]
    if c <= 4:
        modes.append((_abi.RL_NCHW_NCHW4_IC_SMALL, _abi.RL_NCHW4_NCHW))
    for to, back in modes:
        y = ops.relayout_exec(ops.relayout_desc(to, x.shape), to_dev(x))
        z = torch.full(x.shape, 55, dtype=torch.int8, device="cuda")
        ops.relayout_exec(ops.relayout_desc(back, tuple(y.shape), oc=c), y, z)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), oracle.relayout(oracle.relayout_desc(to, x.shape), x)), to
        assert np.array_equal(z.cpu().numpy(), x), back


@pytest.mark.parametrize("h,w", [(1, 1), (3, 5), (8, 8), (13, 29)])
def test_packed_to_packed(oracle, h, w):
    x = util.uniform_int(h * 100 + w, (3, 16, h, w, 4), -128, 127, np.int8)
    y = ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW4_NCHW32, x.shape), to_dev(x))
    back = ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW32_NCHW4, tuple(y.shape)), y)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), oracle.relayout(oracle.relayout_desc(_abi.RL_NCHW4_NCHW32, x.shape), x))
    assert np.array_equal(back.cpu().numpy(), x)


@pytest.mark.parametrize("window,stride,pad,size", [((4, 4), 4, 0, (9, 8)), ((1, 17), 1, (0, 3), (2, 20)), ((7, 7), 7, 0, (7, 7)),
                                                    ((9, 9), 9, 0, (9, 9)), ((5, 5), 2, 2, (8, 7)), ((33, 31), 1, 16, (33, 31))])
@pytest.mark.parametrize("fmt,c", [("NCHW", 7), ("NCHW4", 12), ("NCHW32", 96)])
@pytest.mark.parametrize("mode", ["MAX", "AVERAGE", "AVERAGE_COUNT_EXCLUDE_PADDING"])
def test_large_windows(oracle, mode, fmt, c, window, stride, pad, size):
    d = _abi.make_pooling_desc(mode, fmt, 3, c, size[0], size[1], window, stride, pad)
    x = util.uniform_int(sum(window) + c, _abi.packed_shape(d.format, 3, c, *size), -128, 127, np.int8)
    got = ops.pooling_exec(d, to_dev(x))
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), oracle.pooling(d, x))


# Tensors beyond 2 GiB (offsets in 64 bits) and beyond 4 GiB (one thread per byte would be more threads than a launch can
# number): planes of whole and of broken 16-byte vectors, and planes too small for either kernel of vectors
@pytest.mark.parametrize("shape", [(9, 64, 2048, 2048), (9, 63, 1999, 2003), (33000, 97, 26, 27), (44000, 1030, 7, 7),
                                   (17, 64, 2048, 2048)])
def test_large_tensors(shape):
    n, c, h, w = shape
    x = torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda")
    assert x.numel() >= 1 << 31
    for to, back, p in ((_abi.RL_NCHW_NCHW4, _abi.RL_NCHW4_NCHW, 4), (_abi.RL_NCHW_NCHW32, _abi.RL_NCHW32_NCHW, 32)):
        y = ops.relayout_exec(ops.relayout_desc(to, shape), x)
        assert y.shape == (n, -(-c // p), h, w, p)
        for lo in range(0, n, max(1, n // 8)):
            part = y[lo:lo + max(1, n // 8)].permute(0, 1, 4, 2, 3).reshape(-1, y.shape[1] * p, h, w)
            assert torch.equal(part[:, :c], x[lo:lo + part.shape[0]]), (p, lo)
            assert not part[:, c:].any(), (p, lo)
        z = ops.relayout_exec(ops.relayout_desc(back, tuple(y.shape), oc=c), y)
        assert torch.equal(z, x), p
        del y, z
    if c % 32 == 0:
        y = x.view(n, c // 4, h, w, 4)
        z = ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW4_NCHW32, tuple(y.shape)), y)
        for lo in range(n):
            assert torch.equal(z[lo].view(c // 32, h * w, 8, 4).permute(0, 2, 1, 3).reshape(c // 4, h, w, 4), y[lo]), lo
        assert torch.equal(ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW32_NCHW4, tuple(z.shape)), z), y)


@pytest.mark.parametrize("n,c,h,w", [(9, 5, 1031, 481), (9, 3, 1031, 481), (4096, 4, 33, 31), (2, 12, 3, 700001), (1, 4, 2048, 2047), (1, 4, 2048, 2048)])
def test_nchw4_with_several_steps_to_a_thread(n, c, h, w):
    """Both sides of the line (2^22 pixels of a channel block in all), last steps that overlap and threads with a part of their
    steps.  A layout conversion moves bytes, so torch's own copies are the reference."""
    x = torch.randint(-128, 128, (n, c, h, w), dtype=torch.int8, device="cuda")
    blocks = (c + 3) // 4
    want = torch.zeros((n, blocks * 4, h, w), dtype=torch.int8, device="cuda")
    want[:, :c] = x
    want = want.view(n, blocks, 4, h, w)
    y = ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW_NCHW4_IC_SMALL if c < 4 else _abi.RL_NCHW_NCHW4, (n, c, h, w)), x)
    assert torch.equal(y, want.permute(0, 1, 3, 4, 2))
    back = ops.relayout_exec(ops.relayout_desc(_abi.RL_NCHW4_NCHW, tuple(y.shape)), y)
    assert torch.equal(back, want.reshape(n, blocks * 4, h, w))
