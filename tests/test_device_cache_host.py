"""CPU: the device memory kept for reuse, over a stub of the HIP library."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_device_cache_under_host_allocation_failures(tmp_path):
    """Memory released while host memory runs out is freed or kept, never both,
    and none is lost; what is kept stays within its bound."""
    host = os.path.join(ROOT, "gaffa_amd", "csrc", "host")
    exe = str(tmp_path / "device_cache")
    subprocess.run(["g++", "-std=c++20", "-O1", "-I" + os.path.join(ROOT, "include"), "-I" + host,
                    os.path.join(ROOT, "tests", "native", "device_cache.cpp"),
                    os.path.join(host, "hip_runtime.cpp"), "-o", exe, "-pthread"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout + run.stderr
