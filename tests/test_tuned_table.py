"""The tuned table's measurements are the tuner's own: each entry's rate is its shape's operations over its time."""

import json

import pytest

from kernel_library.config import TUNED_TABLE


def test_rates_follow_from_times():
    doc = json.loads(TUNED_TABLE.read_text())
    assert doc["measurements"].keys() <= doc["configs"].keys()
    for key, m in doc["measurements"].items():
        M, N, K = map(int, key.split(":")[1].split("x"))
        assert m["tflops"] == pytest.approx(2.0 * M * N * K / m["total_time_s"] / 1e12, rel=1e-12), key
