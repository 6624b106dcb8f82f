"""The library's memory layer on the CPU: csrc/common.hpp and csrc/memory.cpp compiled with the host compiler against
stand-ins for the HIP calls (tests/host_memory.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_memory") / "host_memory")
    subprocess.run(["g++", "-std=c++17", "-g", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "host_memory.cpp"), "-o", exe, "-pthread"], check=True)
    return exe


@pytest.mark.parametrize("what", ["staging_readback", "failed_allocation", "capacity"])
def test_memory_layer(checks, what):
    r = subprocess.run([checks, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
