"""The bytes behind bench.py's roofline: what no launch can do without is no more
than what the counters of the recorded profiles saw."""
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402

CELLS = 4096 * 4096


def test_least_bytes_are_below_the_counted_traffic():
    with open(os.path.join(ROOT, "profiles", "traffic.json")) as fh:
        counted = json.load(fh)
    # kernel -> storage, steps per launch
    for key, (storage, k) in {"k_step_f32_periodic_fluid_4096": ("f32", 1), "k_step_f16_periodic_fluid_4096": ("f16", 1),
                              "k_step_tb_f32_periodic_fluid_4096": ("f32", 8),
                              "k_step_ts_f32_periodic_fluid_4096": ("f32", 8)}.items():
        least = k * CELLS * bench.step_bytes_per_cell(storage, k)
        assert 0.6 * counted[key] < least <= counted[key], key
    # the two 8-step kernels have a figure each: regions read their halo, strips less of it
    assert counted["k_step_ts_f32_periodic_fluid_4096"] < counted["k_step_tb_f32_periodic_fluid_4096"]
    # 2048^2 FP64, profiles/k_step_ts.md
    assert 8 * 2048 * 2048 * bench.step_bytes_per_cell("f64", 8) < 725.7e6


def test_a_runs_bytes_follow_its_launches():
    for storage, k, steps, launches in (("f32", 8, 20, 3), ("f32", 8, 19, 5), ("f32", 8, 1000, 125), ("f64", 8, 13, 3),
                                        ("f16", 8, 20, 6), ("f32", 1, 20, 20), ("f32", 4, 7, 4)):
        assert bench.launched_bytes_per_cell(storage, k, steps) == bench.BYTES_PER_CELL[storage] * launches / steps
