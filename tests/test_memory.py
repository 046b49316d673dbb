"""Bookkeeping of device memory (hom3_amd/csrc/memory.hpp): what the adjoint's
workspace takes at the limit of a device, over calls of many sizes, and what
becomes of the memory kept between calls when another allocation runs short.
Host-only: tests/cpp/memory_check.cpp is compiled with g++ against a stand-in
for the HIP allocation calls."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_device_memory_bookkeeping(tmp_path):
    exe = str(tmp_path / "memory_check")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", os.path.join(HERE, "cpp", "host_stub"),
           "-I", os.path.join(ROOT, "hom3_amd", "csrc"), os.path.join(HERE, "cpp", "memory_check.cpp"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-3000:]
