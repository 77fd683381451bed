"""Figures that bench.py derives on the host (CPU)."""
from types import SimpleNamespace

import torch

import bench


def test_missed_rows_counts_rows_and_not_blocks():
    """Two full blocks and a last one of three rows, then one of one row; what lies past a group's count is left over
    from an earlier step."""
    sizes = torch.tensor([[8, 8, 3, 8, 5], [1, 8, 8, 8, 8], [7, 7, 7, 7, 7]], dtype=torch.int32)
    cache = SimpleNamespace(miss_unit_sizes=[None, sizes], miss_num_units=[None, torch.tensor([3, 1, 0], dtype=torch.int32)])
    assert bench.missed_rows(cache, 1) == 8 + 8 + 3 + 1
