"""LDS by which the lanes of one wave hand data to each other (no GPU): the front end's code for the kernels that do so holds the fence and
the wave barrier of lds_between_lanes between the stores of one lane and the loads of another, and between those and the next stores.
Without them the compiler may swap the two wherever it can tell that a lane's own addresses differ, which no run shows until it does."""
import os
import re
import subprocess

import pytest

from megengine_amd import build

CALL = "lds_between_lanes"


def _functions(source):
    ir = subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-w", "-Xclang", "-disable-llvm-passes", "-S",
                         "-emit-llvm", "--offload-device-only", os.path.join(build.CSRC, source), "-o", "-"],
                        capture_output=True, text=True, check=True).stdout
    return {re.search(r"@([\w$.]+)\(", f).group(1): f for f in re.findall(r"^define [^\n]*\n.*?^}", ir, re.S | re.M)}


def _parts(body):
    return re.split(r"call [^\n]*%s[^\n]*" % CALL, body)


@pytest.fixture(scope="module")
def split():
    return _functions("conv_igemm5.hip")


def test_the_fence_orders_memory_and_lanes(split):
    body = next(f for name, f in split.items() if CALL in name)
    at = [body.index(s) for s in ('fence syncscope("wavefront") release', "llvm.amdgcn.wave.barrier", 'fence syncscope("wavefront") acquire')]
    assert at == sorted(at)


def test_filter_rows_turned_in_lds(split):
    # the stage of ks_run<.., TURN = true, ..>: the lambda that multiplies and loads both operands again
    stages = [f for name, f in split.items() if re.search(r"6ks_runI\w+ELb1ENS0_6Ks(Wire|Wide)E\w*ENKUl", name) and "mfma" in f]
    assert len(stages) >= 16
    for f in stages:
        parts = _parts(f)
        assert len(parts) == 3, f.split("\n")[0]
        assert "store <4 x i32>" in parts[0] and "mfma" not in parts[0]     # rows into LDS
        assert "load <4 x i32>" in parts[1] and "mfma" not in parts[1]      # operands out of it
        assert "store <4 x i32>" not in parts[2] and "mfma" in parts[2]


def test_bias_of_a_wave():
    runs = [f for name, f in _functions("conv_pw4.hip").items() if "8pw4q_runI" in name and CALL in f]
    assert len(runs) >= 8
    for f in runs:
        assert len(_parts(f)) == 2, f.split("\n")[0]
