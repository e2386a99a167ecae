"""Host checks (no GPU) of the renderer: tests/renderer_host_check.cpp
with the library's host code over host memory (tests/fake_hip.h)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ataraxia_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not shutil.which("g++") or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("needs g++ and the ROCm headers")
    exe = tmp_path_factory.mktemp("renderer_host") / "check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{CSRC}", os.path.join(ROOT, "tests", "renderer_host_check.cpp"),
                    *(os.path.join(CSRC, f"{n}.cpp") for n in ("renderer", "host_common", "host_transfer", "bvh_build")),
                    "-lpthread", "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("name", ["upload", "devices"])
def test_renderer(check, name):
    out = subprocess.run([check, name], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and "all checks passed" in out.stdout, out.stderr
