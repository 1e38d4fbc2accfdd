"""bench.py's figures per batch size: which kernel's committed counters they
come from, and that every size it reports has them."""

from __future__ import annotations

import pytest

import bench

RUN = {"kernel_ms_per_launch": 2.7, "env_steps_per_s": 1.5e6, "instructions_per_env_step": 31150.0}


def test_small_batches_take_the_counters_of_their_own_kernel():
    f = bench.size_figures(RUN, 4096)
    assert f["consoles_per_wave"] == 1
    # One console in scalar registers: lanes are no measure of its use.
    assert f["useful_lane_frac"] is None and f["useful_valu_lane_ops_frac"] is None
    assert 0 < f["valu_busy_frac"] < 1 and 0 < f["salu_busy_frac"] < 1
    assert 0 < f["valu_lane_ops_frac"] < f["valu_busy_frac"]
    # About 10 KB of HBM traffic per env-step, twice what a step must move.
    assert f["hbm_algorithmic_gbs"] < f["hbm_measured_gbs"] < 3 * f["hbm_algorithmic_gbs"]


def test_the_full_batch_takes_the_lane_kernels():
    f = bench.size_figures({**RUN, "kernel_ms_per_launch": 18.8}, 65536)
    assert f["consoles_per_wave"] == 64 and f["useful_lane_frac"] == 1.0
    assert f["valu_busy_frac"] == pytest.approx(0.5676) and f["salu_busy_frac"] < 0.2
    assert f["useful_valu_lane_ops_frac"] == f["valu_lane_ops_frac"]


def test_sizes_without_counters_report_none():
    f = bench.size_figures(RUN, 5000)
    assert f["valu_busy_frac"] is None and f["hbm_measured_gbs"] is None
