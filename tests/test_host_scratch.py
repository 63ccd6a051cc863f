"""The library's scratch bookkeeping (csrc/wq_scratch.cpp) compiled for the CPU against stand-ins of the HIP calls."""
import os
import shutil
import subprocess

import pytest

from _lib import ROOT

CSRC = os.path.join(ROOT, "agens-engine_amd", "csrc")


def test_scratch_bookkeeping(tmp_path):
    gxx, rocm = shutil.which("g++"), os.environ.get("ROCM_PATH", "/opt/rocm")
    if not gxx or not os.path.exists(os.path.join(rocm, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "test_scratch")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(rocm, "include"), "-I" + CSRC, os.path.join(CSRC, "wq_scratch.cpp"),
                    os.path.join(ROOT, "tests", "host", "test_scratch.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
