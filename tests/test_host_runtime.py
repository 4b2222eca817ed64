"""The host side of contexts, the block memory pool and the staged copies, without a GPU: tests/c/host_runtime.cpp compiles
the library's own sources against a HIP runtime of plain memory that counts allocations and keeps the last error."""
import glob
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "high-order-accurate-cfd-solver-code-for-heterogenous-hardware-cpu-and-gpgpu-_amd", "csrc")
HIP_INCLUDE = next(iter(glob.glob("/opt/rocm/include/hip/hip_runtime.h")), None)


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None or HIP_INCLUDE is None:
        pytest.skip("g++ or the HIP headers not available")
    exe = str(tmp_path_factory.mktemp("host") / "host_runtime")
    cmd = ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC,
           os.path.join(ROOT, "tests", "c", "host_runtime.cpp")]
    cmd += [os.path.join(CSRC, f) for f in ("ctx.cpp", "host_copy.cpp", "common.cpp")] + ["-lpthread", "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("check", ["pool", "trim", "pinned", "rings"])
def test_host_runtime(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
