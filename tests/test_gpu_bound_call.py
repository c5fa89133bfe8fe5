"""Bound ConvBias calls (mi355_convbias_s8_bind through ops.conv_bias_bind): a replay reads the tensors as they are when it
runs, covers the algorithms that launch one kernel, several kernels or use a workspace, and a call that exec would refuse
is refused when it is called."""
import numpy as np
import pytest
import torch

from megengine_amd import _abi, lib, ops
from tests import util

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
CASES = [
    dict(fmt="NCHW32", n=2, ic=64, ih=9, iw=11, oc=96, fh=3, pad=1, has_z=True),
    dict(fmt="NCHW4", n=3, ic=24, ih=10, iw=12, oc=24, fh=3, group=3, pad=1),
    dict(fmt="NCHW4", n=2, ic=32, ih=9, iw=9, oc=32, fh=5, group=32, pad=2),
    dict(fmt="NCHW", n=2, ic=40, ih=23, iw=19, oc=37, fh=3, pad=1, has_z=True),
    dict(fmt="NCHW4", n=1, ic=4, ih=30, iw=30, oc=16, fh=7, pad=3, stride=2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(CASES)))
def test_bound_call_equals_exec_on_every_replay(oracle, i):
    c = dict(CASES[i])
    d = _abi.make_conv_desc(c.pop("fmt"), c.pop("n"), c.pop("ic"), c.pop("ih"), c.pop("iw"), c.pop("oc"), c.pop("fh"),
                            nonline="RELU", **c, **S)
    algo, ws = ops.conv_bias_query(d)
    first = util.make_tensors(d, seed=70 + i)
    dev = [None if x is None else torch.from_numpy(x).cuda() for x in first]
    dst = torch.full(_abi.conv_shapes(d)[3], 77, dtype=torch.int8, device="cuda")
    work = torch.empty(ws, dtype=torch.uint8, device="cuda") if ws else None
    side = torch.cuda.Stream()
    call = ops.conv_bias_bind(d, *dev, dst, algo, workspace=work)
    on_side = ops.conv_bias_bind(d, *dev, dst, algo, workspace=work, stream=side.cuda_stream)
    for k, run in enumerate((call, on_side, call)):
        host = first if k == 0 else util.make_tensors(d, seed=170 + 10 * k + i)
        for t, x in zip(dev, host):
            if t is not None:
                t.copy_(torch.from_numpy(x))
        dst.fill_(77)
        torch.cuda.synchronize()
        run()
        torch.cuda.synchronize()
        assert np.array_equal(dst.cpu().numpy(), oracle.conv_bias(d, *host)), (i, k)


@pytest.mark.gpu
def test_bound_call_that_exec_refuses_raises_when_called():
    d = _abi.make_conv_desc("NCHW4", 2, 64, 9, 9, 64, 3, pad=1, nonline="RELU", **S)
    src, flt, bias, _ = [None if x is None else torch.from_numpy(x).cuda() for x in util.make_tensors(d, seed=3)]
    dst = torch.empty(_abi.conv_shapes(d)[3], dtype=torch.int8, device="cuda")
    algo, _ = ops.conv_bias_query(d, lib.algo_names().index("MI355_IGEMM_MFMA_I8"))
    algo.tile_cfg = lib.tile_names().index("v2_128x128x64r4")  # no tile of this problem
    call = ops.conv_bias_bind(d, src, flt, bias, None, dst, algo)
    with pytest.raises(lib.Mi355Error) as e:
        call()
    assert e.value.status == _abi.ERR_ALGO


def test_arguments_are_checked_without_a_gpu():
    d = _abi.make_conv_desc("NCHW4", 1, 8, 4, 4, 8, 1)
    x = torch.zeros(1, 2, 4, 4, 4, dtype=torch.int8)
    with pytest.raises(RuntimeError):
        ops.conv_bias_bind(d, x, x, None, None, x, ops.conv_bias_query(d)[0])
    with pytest.raises(TypeError):
        ops.conv_bias_exec(d, src=x)
    with pytest.raises(TypeError):
        ops.conv_bias_exec(d, x, x, nothing=1)
    with pytest.raises(TypeError):
        ops.conv_bias_exec(d, x, x, src=x)
    with pytest.raises(KeyError):
        ops.elemwise_q_exec("SIGMOID", [x], [1.0], 1.0)
    with pytest.raises(RuntimeError):
        ops.requant_exec(x.to(torch.float32), 1.0, 1.0)
