"""The dataset memory's host logic (tuvok_amd/csrc/devmem.cpp), compiled with g++ over
a pretended device and run on the CPU: what it does when the device is full."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_devmem_on_a_full_device(tmp_path):
    exe = tmp_path / "devmem_check"
    cpp = os.path.join(ROOT, "tests", "cpp")
    csrc = os.path.join(ROOT, "tuvok_amd", "csrc")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(cpp, "fakehip"), "-I", csrc,
                        os.path.join(cpp, "devmem_check.cpp"), os.path.join(csrc, "devmem.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
