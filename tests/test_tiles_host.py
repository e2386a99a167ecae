"""Host-side check of the tile queries (no GPU): tests/tile_check.cpp builds
tiles with ataraxia_amd/csrc/bvh_build.cpp and runs a float restatement of the
device query against the oracle's flat closest-hit loop (ora_trace_ray)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FLAGS = ["-O2", "-ffp-contract=off", "-fno-fast-math"]


def test_tile_queries_match_flat_loop(tmp_path):
    if not shutil.which("g++") or not shutil.which("gcc"):
        pytest.skip("no host C/C++ compiler")
    ora, exe = tmp_path / "oracle.o", tmp_path / "tile_check"
    subprocess.run(["gcc", "-std=c99", *FLAGS, "-c", os.path.join(ROOT, "oracle", "atx_oracle.c"), "-o", str(ora)],
                   check=True)
    subprocess.run(["g++", "-std=c++17", *FLAGS, os.path.join(ROOT, "tests", "tile_check.cpp"),
                    os.path.join(ROOT, "ataraxia_amd", "csrc", "bvh_build.cpp"), str(ora), "-lm", "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe), "12000"], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0, out.stderr
    assert len(out.stdout.splitlines()) == 15
