"""Host-side check (no GPU) of tile queries over tiles as the library builds them:
tests/tile_production_check.cpp, optimised and under the sanitizers."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FLAGS = ["-ffp-contract=off", "-fno-fast-math"]
SANITIZE = ["-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all"]


@pytest.mark.parametrize("flags,rays", [(["-O2"], "4000"), (SANITIZE, "300")],
                         ids=["optimised", "sanitized"])
def test_tiles_as_built_by_the_library(tmp_path, flags, rays):
    if not shutil.which("g++") or not shutil.which("gcc"):
        pytest.skip("no host C/C++ compiler")
    ora, exe = tmp_path / "oracle.o", tmp_path / "check"
    subprocess.run(["gcc", "-std=c99", *FLAGS, *flags, "-c", os.path.join(ROOT, "oracle", "atx_oracle.c"),
                    "-o", str(ora)], check=True)
    subprocess.run(["g++", "-std=c++17", *FLAGS, *flags, os.path.join(ROOT, "tests", "tile_production_check.cpp"),
                    os.path.join(ROOT, "ataraxia_amd", "csrc", "bvh_build.cpp"), str(ora), "-lm", "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe), rays], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr
    assert len(out.stdout.splitlines()) == 16 and "spheres=17001" in out.stdout
