"""The tuned table's measurements: each rate is its shape's operations over its time (some entries are kept with the
digits a table prints, so within 0.5 %), and the fp32 entry holds a time of the tuner, which launches one call at a
time and so never reads less than a launch and a kernel (calls back to back take 4.4 us there)."""

import json

import pytest

from kernel_library.config import TUNED_TABLE


def _measured():
    doc = json.loads(TUNED_TABLE.read_text())
    assert doc["measurements"].keys() <= doc["configs"].keys()
    return doc["measurements"]


def test_rates_follow_from_times():
    for key, m in _measured().items():
        M, N, K = map(int, key.split(":")[1].split("x"))
        assert m["tflops"] == pytest.approx(2.0 * M * N * K / m["total_time_s"] / 1e12, rel=5e-3), key


def test_the_fp32_entry_is_a_time_of_the_tuner():
    assert _measured()["matmul_lhsT_rhs_f32:256x512x512"]["total_time_s"] > 7e-6
