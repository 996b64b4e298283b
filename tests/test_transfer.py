"""Host transfers from a thread whose current device is not the library's: the
library's own source against HIP calls on host memory (transfer_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"),
                    reason="needs g++ and the HIP headers")
def test_host_copy_from_another_device(tmp_path):
    exe = str(tmp_path / "transfer_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "qcd_amd", "csrc"),
                    os.path.join(ROOT, "tests", "transfer_check.cpp"),
                    os.path.join(ROOT, "qcd_amd", "csrc", "transfer.cpp"), "-o", exe, "-lpthread"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
