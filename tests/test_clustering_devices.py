"""A clustering object used under one device after another: the stream and
events that it keeps belong to the device of the call (a stand-in HIP runtime
with two devices, on the CPU)."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_predict_under_another_device(tmp_path):
    if not shutil.which("g++") or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "clustering_devices")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "pyglass_amd", "csrc"),
                    os.path.join(ROOT, "tests", "clustering_devices.cpp"),
                    os.path.join(ROOT, "pyglass_amd", "csrc", "clustering.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"exit {r.returncode}: {r.stdout}"
