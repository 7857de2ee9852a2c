"""The host side's device-memory pool where memory runs short, on a stand-in runtime (tests/cpp/pool_check.cpp): idle
temporaries go back and the allocation succeeds without leaving an error for the check after the next launch."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(__file__)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(f"{ROCM}/include/hip"), reason="needs g++ and HIP's headers")
def test_allocations_when_memory_runs_short(tmp_path):
    exe = tmp_path / "pool_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", "-o", str(exe),
                    f"{HERE}/cpp/pool_check.cpp", "-lpthread"], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
