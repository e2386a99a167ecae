"""Host-side check (no GPU) of the shading's quotients from inexact starts:
tests/quotient_check.cpp against the compiler's."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_quotients_from_starts_one_ulp_off(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "quotient_check"
    subprocess.run(["g++", "-std=c++20", "-O2", "-mfma", "-ffp-contract=off", "-fno-fast-math",
                    os.path.join(ROOT, "tests", "quotient_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
