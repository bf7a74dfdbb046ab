"""The library's pool of page-locked memory and its shared host copies (csrc/host_io.h), checked on the CPU by a program
that links the library and brings its own stand-ins for the runtime's two allocation calls (tests/cpp/host_io_test.cpp)."""
import os
import subprocess

import pytest

from fyusenet_amd import build

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "host_io_test.cpp")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_io") / "host_io_test")
    r = subprocess.run([build.HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-Wall", SRC, "-o", exe, "-rdynamic",
                        "-L", build.HERE, "-lfynhip", "-Wl,-rpath," + build.HERE], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("check", ["loans", "runtime_calls_outside_the_lock", "copies_without_helpers"])
def test_host_io(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
