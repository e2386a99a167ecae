"""The benchmark's roofline entries: pairs that matrix products decide are priced
as matrix work, tests on the vector units as vector work."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


STATS = {"sphere_tests": 3_000_000_000, "box_tests": 500_000_000, "launches": 2, "path_ms": 4.0, "rays": 10,
         "reused_rays": 2, "exact_retraces": 1}


def test_tests_on_the_vector_units(bench):
    e = bench.roofline(STATS, None)
    assert e["bound"] == "valu" and e["peak"] == bench.FP32_VALU_PEAK_TFLOPS
    assert e["achieved"] == pytest.approx((17 * 3.0 + 12 * 0.5) / 4.0)   # TFLOP in 4 ms, over 2 launches
    assert e["frac"] == pytest.approx(e["achieved"] / e["peak"])


def test_pairs_of_matrix_products(bench):
    e = bench.roofline({**STATS, "box_tests": 0}, None, products=True)
    assert e["bound"] == "mfma" and e["peak"] == bench.F16_MATRIX_PEAK_TFLOPS
    assert e["achieved"] == pytest.approx(64 * 3.0 / 4.0)
    assert e["frac"] == pytest.approx(e["achieved"] / e["peak"])
