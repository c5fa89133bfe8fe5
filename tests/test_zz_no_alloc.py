"""The allocation-free exec entry point (mi355_convbias_s8_exec_static_workspace) against mi355_convbias_s8_exec.

Collected last on purpose (the file name sorts after every other test file): the suite runs with -x, and a failure here
must not hide the tests of the operator proper."""
import ctypes as C

import numpy as np
import pytest
import torch

from megengine_amd import _abi, lib, ops
from tests import util
from tests.routes import routes

pytestmark = pytest.mark.gpu

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)


def _exec_static(d, algo, src, flt, bias, z, dst):
    return lib.lib().mi355_convbias_s8_exec_static_workspace(
        C.c_void_p(torch.cuda.current_stream().cuda_stream), C.byref(d), None if algo is None else C.byref(algo), ops._ptr(src),
        ops._ptr(flt), ops._ptr(bias), ops._ptr(z), ops._ptr(dst))


def _case(d, seed):
    src, flt, bias, z = util.make_tensors(d, seed=seed)
    return [None if x is None else torch.from_numpy(x).cuda() for x in (src, flt, bias, z)]


@pytest.mark.parametrize("fh,fw,packs", [(5, 3, True), (3, 3, False)])
def test_static_workspace_exec_matches_exec_two_calls_in_a_row(fh, fw, packs):
    """Two calls in a row on the one array, the second with a smaller input (its tensors cover only the front of what
    the first call left behind), then the first again: each must equal mi355_convbias_s8_exec with a workspace of the
    caller's, bit for bit, for the algorithm that needs the workspace (plain NCHW, packed ahead of the MFMA kernel).  The smaller
    layer is packed too, or one that runs in a single launch and touches no workspace."""
    nchw = lib.algo_names().index("MI355_NCHW_RELAYOUT_MFMA_I8")
    big = _abi.make_conv_desc("NCHW", 4, 24, 28, 28, 40, 3, pad=1, nonline="RELU", has_z=True, **S)
    small = _abi.make_conv_desc("NCHW", 2, 20, 19, 23, 36, fh, fw, pad=(fh // 2, fw // 2), nonline="H_SWISH", has_z=True, **S)
    written = {id(big): True, id(small): packs}
    assert [r.kernels[0] == "nchw_prep_kernel" for r in routes([(d, nchw, -1, True) for d in (big, small)])] == [True, packs]
    assert lib.lib().mi355_static_workspace_bytes() == 32 << 20
    plans = []
    for d, seed in ((big, 5), (small, 6)):
        algo, ws = ops.conv_bias_query(d, nchw)
        assert algo.id == nchw and 0 < ws <= lib.lib().mi355_static_workspace_bytes()
        t = _case(d, seed)
        room = torch.full((ws,), 113, dtype=torch.uint8, device="cuda")
        want = ops.conv_bias_exec(d, *t, algo=algo, workspace=room)
        torch.cuda.synchronize()
        assert bool((room != 113).any()) == written[id(d)]
        plans.append((d, algo, t, want))
    for d, algo, t, want in (plans[0], plans[1], plans[0]):
        got = torch.full_like(want, 77)
        assert _exec_static(d, algo, *t, got) == 0, lib.lib().mi355_last_error()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    # without an algorithm the heuristic makes the same choice, inside the array
    d, algo, t, want = plans[1]
    got = torch.full_like(want, 77)
    assert _exec_static(d, None, *t, got) == 0, lib.lib().mi355_last_error()
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_static_workspace_exec_runs_the_other_algorithms_unchanged():
    """Algorithms without a workspace go through the same entry point untouched."""
    d = _abi.make_conv_desc("NCHW32", 2, 64, 14, 14, 64, 3, pad=1, nonline="RELU", has_z=True, **S)
    t = _case(d, 9)
    algo, ws = ops.conv_bias_query(d)
    assert ws == 0
    want = ops.conv_bias_exec(d, *t, algo=algo)
    got = torch.full_like(want, 77)
    assert _exec_static(d, algo, *t, got) == 0, lib.lib().mi355_last_error()
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_static_workspace_exec_refuses_what_does_not_fit():
    """A problem whose workspace exceeds the array: MI355_ERR_WORKSPACE for the algorithm by name, the generic kernel from
    the heuristic; nothing is launched in the first case."""
    nchw = lib.algo_names().index("MI355_NCHW_RELAYOUT_MFMA_I8")
    d = _abi.make_conv_desc("NCHW", 32, 64, 112, 112, 64, 3, pad=1, nonline="RELU", **S)
    algo, ws = ops.conv_bias_query(d, nchw)
    assert ws > lib.lib().mi355_static_workspace_bytes()
    ss, fs, bs, ds = _abi.conv_shapes(d)
    src = torch.zeros(ss, dtype=torch.int8, device="cuda")
    flt = torch.zeros(fs, dtype=torch.int8, device="cuda")
    bias = torch.zeros(bs, dtype=torch.int32, device="cuda")
    dst = torch.full(ds, 77, dtype=torch.int8, device="cuda")
    assert _exec_static(d, algo, src, flt, bias, None, dst) == _abi.ERR_WORKSPACE
    assert "static workspace" in lib.lib().mi355_last_error().decode()
    torch.cuda.synchronize()
    assert int((dst != 77).sum()) == 0


def test_exec_that_chooses_for_itself_goes_by_what_is_written():
    """Without an algorithm, a workspace that holds the packed src and filter is enough for the plain-NCHW algorithm, although
    query reports more and exec asks a caller who names it for that; with less the generic kernel leaves it alone."""
    L, names = lib.lib(), lib.algo_names()
    up = lambda x: (x + 255) // 256 * 256
    d = _abi.make_conv_desc("NCHW", 4, 24, 28, 28, 40, 3, pad=1, nonline="RELU", has_z=True, **S)
    used = up(4 * 32 * 28 * 28) + up(40 * 32 * 9)
    t = [torch.from_numpy(x).cuda() for x in util.make_tensors(d, seed=5)]
    algo, ws = ops.conv_bias_query(d)
    assert names[algo.id] == "MI355_NCHW_RELAYOUT_MFMA_I8" and ws > used
    want = ops.conv_bias_exec(d, *t)
    for size, shift, written in ((used, 0, True), (used - 1, 0, False), (ws - 16, 4, False)):
        buf = torch.full((used + ws + 256,), 113, dtype=torch.uint8, device="cuda")
        dst = torch.zeros_like(want)
        args = [ops._ptr(x) for x in t] + [ops._ptr(dst), ops._ptr(buf[shift:]), size]
        assert L.mi355_convbias_s8_exec(ops._stream(), d, None, *args) == 0, L.mi355_last_error()
        torch.cuda.synchronize()
        assert torch.equal(dst, want)
        assert bool((buf != 113).any()) == written
        assert bool((buf[shift + size:] == 113).all())
        assert L.mi355_convbias_s8_exec(ops._stream(), d, algo, *args) == _abi.ERR_WORKSPACE
