"""bench.py's roofline figures are rates of what the timed kernel moves."""
from __future__ import annotations

import json
from pathlib import Path

import pytest

import bench

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.parametrize("ms", [0.25, 0.5842])
def test_roofline_is_the_profiled_traffic_over_the_launch(ms):
    profile = json.loads((ROOT / "profiles" / "closest_hit_traffic.json").read_text())
    r = bench.roofline(ms, profile["hbm_bytes_per_launch"])
    assert r["kernel"] == profile["kernel"]
    assert r["achieved"] == pytest.approx(profile["hbm_bytes_per_launch"] / ms / 1e6, abs=0.1)
    assert r["frac"] == pytest.approx(r["achieved"] / r["peak"], abs=1e-4)
    assert profile["hbm_bytes_per_launch"] == profile["read_bytes_per_launch"] + profile["write_bytes_per_launch"]


def test_roofline_of_a_form_without_a_traffic_profile():
    assert bench.roofline(0.5, None)["achieved"] is None
    r = bench.roofline(0.5, 10 ** 9, ray_windows=1)
    assert r["kernel"] == "k_closest_hit" and r["traffic"] is None and r["frac"] is None
