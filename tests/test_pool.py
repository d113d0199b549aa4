"""Device blocks kept between objects, on the host: given back when an
allocation of any size finds no memory, and with the last context."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"),
                    reason="needs g++ and the HIP headers")
def test_kept_blocks_on_the_host(tmp_path):
    exe = str(tmp_path / "pool_check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Iinclude",
                        "tests/pool_check.cpp", "the-tessellator_amd/csrc/pool.cpp", "-o", exe], cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "as stated" in r.stdout, r.stdout + r.stderr
