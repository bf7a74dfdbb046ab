"""Layers whose packed weights are larger than a kernel's 32-bit offsets reach go to another form of the convolution, checked
on the CPU by a program that links the library (tests/cpp/weight_offsets_test.cpp)."""
import os
import subprocess

import pytest

from fyusenet_amd import build

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "weight_offsets_test.cpp")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("weight_offsets") / "weight_offsets_test")
    r = subprocess.run([build.HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-Wall", SRC, "-o", exe,
                        "-L", build.HERE, "-lfynhip", "-Wl,-rpath," + build.HERE], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("check", ["p16_rows", "h16"])
def test_weight_offsets(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
