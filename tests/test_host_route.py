"""The host library's choice of the prefill route (host/agens_linear.cpp) on the CPU, against a C ABI that records."""
import os
import shutil
import subprocess

import pytest

from _lib import ROOT

HOST = os.path.join(ROOT, "agens-engine_amd", "host")


def test_prefill_route(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("needs g++")
    exe = str(tmp_path / "test_route")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-I" + os.path.join(ROOT, "include"), "-I" + HOST,
                    os.path.join(HOST, "agens_linear.cpp"), os.path.join(ROOT, "tests", "host", "test_route.cpp"),
                    "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
