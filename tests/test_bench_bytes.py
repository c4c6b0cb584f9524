"""Bytes that bench.py holds a kernel's launches to: one state pass per launch, images and traces once
per step; with one step per launch the specified algorithm's figures."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.parametrize("kernel,launches,steps,calls,expect", [
    ("ac_fwd_step", 8, 8, {"forward": 8}, 24 * 8),
    ("ac_fwd_step", 8, 8, {"recompute": 8}, 28 * 8),
    ("ac_adj_step", 8, 8, {"adjoint": 8}, 28 * 8),
    ("ac_fwd_pair", 4, 8, {"forward+images": 8}, 24 * 4 + 4 * 8),
    ("ac_fwd_tile", 4, 16, {"forward": 8, "recompute": 8}, 24 * 4 + 4 * 8),
    ("ac_adj_tile", 4, 15, {"adjoint": 15}, 24 * 4 + 4 * 15),
    ("el_fwd_step", 8, 8, {"recompute": 8}, 80 * 8),
    ("el3_adj_step", 8, 8, {"adjoint": 8}, 120 * 8),
    ("el_abl_adj", 8, 8, {"adjoint": 8}, 60 * 8),
    ("el_fwd_tile", 4, 8, {"forward": 4, "forward+trace": 4}, 80 * 4 + 20 * 4),
    ("el_adj_tile", 4, 8, {"adjoint": 8}, 80 * 4 + 20 * 8),
    ("abl_fwd_tile", 4, 8, {"recompute": 8}, 20 * 4 + 20 * 8),     # every state written, every second read
    ("abl_adj_tile", 4, 8, {"adjoint": 8}, 40 * 4 + 20 * 8),
])
def test_launch_bytes(kernel, launches, steps, calls, expect):
    import bench
    assert bench.launch_bytes(kernel, launches, steps, calls) == expect
