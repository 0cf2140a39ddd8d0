"""Host threads and the pinned pool of the copies (csrc/hostcopy.hpp), without a GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_threads_and_pool(tmp_path):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("g++ or the HIP headers not installed")
    exe = str(tmp_path / "driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "nflow-red-poplar_amd", "csrc"),
                    os.path.join(ROOT, "tests", "hostcopy_driver.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "threads ok\npool ok\n", (r.returncode, r.stdout, r.stderr)
