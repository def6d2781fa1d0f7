"""The engine's host code (csrc/engine.cpp) on the CPU against a HIP runtime that runs nothing (tests/host/fake_hip.h): the order of
allocations, launches and copies of a call, and what happens where memory does not suffice."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = "/opt/rocm/llvm/bin/clang++"  # (_Float16)
CSRC = os.path.join(ROOT, "strands-decider-web_amd", "csrc")

pytestmark = pytest.mark.skipif(not os.path.exists(CXX), reason="clang++ is missing")


@pytest.fixture(scope="module")
def engine(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    flags = ["-O1", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC]
    r = subprocess.run([CXX] + flags + ["-Wno-unused-result", "-c", os.path.join(CSRC, "engine.cpp"), "-o", str(d / "engine.o")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return d, flags


@pytest.mark.parametrize("name", ["snapshot_order", "gqa_scratch"])
def test_host(engine, name):
    d, flags = engine
    src = os.path.join(ROOT, "tests", "host", name + ".cpp")
    r = subprocess.run([CXX] + flags + ["-Wno-unused-result", "-Wno-unused-function", src, str(d / "engine.o"), "-o", str(d / name), "-lpthread"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(d / name)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
