"""The short exact division over every numerator it is used with, against the
IEEE one on the device (tests/cpp/arith_range_check.cpp, always built from the
present core.h)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


def test_small_numerators():
    subprocess.run(["make", "-C", CPP, "arith_range_check"], check=True, capture_output=True)
    r = subprocess.run([os.path.join(CPP, "arith_range_check")], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
