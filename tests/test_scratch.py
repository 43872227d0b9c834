"""The rules of the library's scratch block (csrc/arena.hpp), on the CPU: the
scenarios of tests/cpp/scratch.cpp, built with g++ over host memory."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    exe = str(tmp_path_factory.mktemp("scratch") / "scratch")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall",
                    "-I", os.path.join(ROOT, "stablediffusion-cpp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "scratch.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["held", "exhausted", "refused", "in_place", "graphs"])
def test_scratch(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
