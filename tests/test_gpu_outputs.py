"""Outputs that an operator allocates by itself: whoever watches or changes torch's allocations meets them too (a dispatch mode, a
profiler, the fill of new memory in deterministic runs)."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from megengine_amd import _abi, ops
from tests import util

pytestmark = pytest.mark.gpu
S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)


def _call(gap=0):
    """a convolution's output and what lies between its images"""
    d = _abi.make_conv_desc("NCHW4", 3, 16, 9, 11, 20, 3, pad=1, nonline="RELU", **S)
    t = [torch.from_numpy(x).cuda() for x in util.make_tensors(d, seed=4)[:3]]
    size = 20 * 9 * 11
    d.dst_stride_n = size + gap if gap else 0
    return lambda: ops.conv_bias_exec(d, *t).view(3, -1), size


def test_dispatch_mode_sees_the_allocation():
    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    call, _ = _call()
    want = call()
    with Log():
        got = call()
    assert any(f.startswith("aten.empty") for f in seen), seen
    assert torch.equal(got, want)


def test_profiler_records_the_allocation():
    call, _ = _call()
    want = call()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as p:
        got = call()
    assert "aten::empty" in [e.key for e in p.key_averages()]
    assert torch.equal(got, want)


def test_deterministic_runs_fill_what_the_operator_leaves():
    call, size = _call(gap=64)
    want = call()[:, :size].clone()
    torch.full((3 * (size + 64),), 5, dtype=torch.int8, device="cuda")  # (freed at once: what the allocator hands out next)
    torch.use_deterministic_algorithms(True)
    try:
        fill = torch.empty(64, dtype=torch.int8, device="cuda")
        got = call()
    finally:
        torch.use_deterministic_algorithms(False)
    assert torch.equal(got[:, :size], want)
    assert bool((fill == fill[0]).all()) and bool((got[:, size:] == fill[0]).all())
