"""Figures that bench.py derives on the host (CPU)."""
import json
from types import SimpleNamespace

import torch

import bench


def test_missed_rows_counts_rows_and_not_blocks():
    """Two full blocks and a last one of three rows, then one of one row; what lies past a group's count is left over
    from an earlier step."""
    sizes = torch.tensor([[8, 8, 3, 8, 5], [1, 8, 8, 8, 8], [7, 7, 7, 7, 7]], dtype=torch.int32)
    cache = SimpleNamespace(miss_unit_sizes=[None, sizes], miss_num_units=[None, torch.tensor([3, 1, 0], dtype=torch.int32)])
    assert bench.missed_rows(cache, 1) == 8 + 8 + 3 + 1


def test_drifting_queries_are_timed_in_whole_rounds_of_their_pool():
    for steps, layers in ((16, 2), (128, 2), (640, 28), (1, 1)):
        untimed, timed = bench.drift_cycles(steps, layers)
        assert untimed >= 16 and untimed % 8 == 0 and timed >= 8 and timed % 8 == 0


def test_traffic_is_of_the_launches_that_the_step_makes(monkeypatch, tmp_path):
    """Recorded for every launch of a step's attention, and on the sources at hand, or not reported."""
    assert bench.attending_launches(bench.CONFIGS["c1"]) == ["step_kernel"]
    assert bench.attending_launches(bench.CONFIGS["c4"]) == ["dist_kernel", "select_attend_kernel"]
    assert bench.attending_launches(bench.CONFIGS["c2"]) == ["dist_kernel", "select_attend_kernel"]
    entry = lambda k: dict(fetch_kib=1000.0, fetch_scale=2.0, write_kib=24.0, write_scale=1.0, source="here",  # noqa: E731
                           kernel_source_sha256_16=bench.kernel_source_hash(k))
    path = tmp_path / "traffic.json"
    monkeypatch.setattr(bench, "TRAFFIC_FILE", str(path))
    assert bench.measured_traffic("c2", ["attend_kernel"])[0] is None
    rec = {k: entry(k) for k in bench.KERNEL_SOURCES}
    path.write_text(json.dumps({"c2": rec}))
    assert bench.measured_traffic("c2", ["dist_kernel", "select_attend_kernel"]) == (2 * 2024 * 1024, "here")
    assert bench.measured_traffic("c5", ["attend_kernel"])[0] is None
    rec["dist_kernel"]["kernel_source_sha256_16"] = "0"
    path.write_text(json.dumps({"c2": rec}))
    assert bench.measured_traffic("c2", ["select_attend_kernel"])[0] and "stale" in bench.measured_traffic("c2", ["dist_kernel"])[1]
