"""Host-side launch planning of libftdx.so on the CPU, under AddressSanitizer + UBSan
(tests/cpp/test_launch_plan.cpp, built with g++ from the library's host-only headers)."""
import os
import shutil
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.mark.skipif(shutil.which("g++") is None or shutil.which("make") is None, reason="needs g++ and make")
def test_launch_plan():
    b = subprocess.run(["make", "-s", "-C", CPP, "test_launch_plan"], capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stdout + b.stderr
    r = subprocess.run([os.path.join(CPP, "test_launch_plan")], capture_output=True, text=True, timeout=600,
                       env=dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0"))
    assert r.returncode == 0 and "ALL PASSED" in r.stdout, r.stdout + r.stderr
