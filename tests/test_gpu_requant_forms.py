"""Stand-alone requantisation around whole rounds of 4096 values to a CU, and counts that four does not divide; every form of the arithmetic, the
literal chain included, for int32 and int8 operands, of which the latter has a loop per form.  Against the oracle."""
import numpy as np
import pytest
import torch

from tests.gpu_util import say
from tests.test_gpu_requant import run_case

pytestmark = pytest.mark.gpu

TILE = 4096


@pytest.mark.parametrize("tiles,more", [(2, -TILE), (2, -TILE + 4), (2, 0), (2, 3), (2, 4), (5, 1023 * 4 + 1), (8, -5), (8, 0), (8, 4)])
def test_sizes(oracle, tiles, more):
    n = tiles * torch.cuda.get_device_properties(0).multi_processor_count * TILE + more
    rng = np.random.RandomState(tiles)
    x, z = rng.randint(-20000, 20000, n).astype(np.int32), rng.randint(-128, 128, n).astype(np.int8)
    say("requant", n)
    run_case(oracle, x, z, 0.0013, 0.17, 0.21, "RELU")
    run_case(oracle, x, None, 0.0013, 0.17, 1.0, "IDENTITY")


@pytest.mark.parametrize("scales", [(0.0013, 0.17, 0.21), (1e-20, 1e-17, 3e-16)])   # a divide-free form; the literal chain
@pytest.mark.parametrize("dtype", [np.int32, np.int8])
def test_forms(oracle, scales, dtype):
    n = 3 * torch.cuda.get_device_properties(0).multi_processor_count * TILE + 77
    rng = np.random.RandomState(1)
    x = rng.randint(-20000, 20000, n).astype(np.int32) if dtype == np.int32 else rng.randint(-128, 128, n).astype(np.int8)
    z = rng.randint(-128, 128, n).astype(np.int8)
    s_src, s_dst, s_z = scales if dtype == np.int32 else (scales[0] * 70, scales[1], scales[2])
    for nl in ("IDENTITY", "RELU", "H_SWISH"):
        say("requant form", nl, dtype.__name__)
        run_case(oracle, x, z, s_src, s_dst, s_z, nl)
        run_case(oracle, x, None, s_src, s_dst, 1.0, nl)
