"""The bench's roofline figures follow the plan that the library reports, not a guess of their own."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


class _Lattice:
    """A stand-in that takes 1 ms a step and runs `plan` steps a launch."""
    plan = 1
    cell_order = 1

    def __init__(self, nx, ny, nz, *a, **k):
        self.fluid_cells = nx * ny * nz

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        pass

    def step_plan(self):
        return self.plan, 64 if self.plan == 2 else 0

    def step_timed(self, n):
        return float(n)

    def tune(self, n):
        return 4

    def measure_copy(self, n, pull=False):
        return float(n)

    def moments(self):
        return np.ones(4)

    def set_flags(self, f):
        pass

    step = init_equilibrium = synchronize = close = lambda self, *a, **k: None


class _Module:
    FP64, FP32_SHIFTED, LAYOUT_TWO_BUFFER, LAYOUT_AA, CELL_ORDER_BRICKS = 0, 1, 0, 1, 2
    Lattice = _Lattice


@pytest.mark.parametrize("plan", [1, 2])
def test_roofline_counts_the_planned_steps_per_launch(plan, monkeypatch):
    monkeypatch.setattr(_Lattice, "plan", plan)
    n, gb = 128, 128 ** 3 * 38 * 8 / 1e9
    r = bench.run_dense(_Module, np.zeros((n, n, n), bool), n, 0.6, 0, 10, 1, 0.0)["roofline"]
    assert r["steps_per_launch"] == plan
    assert r["achieved"] == pytest.approx(gb / (plan * 1e-3), abs=0.06)
    s = bench.run_shard_share(_Module, np.zeros((n, n, n), bool), 0.6, 0.0, planes=4, steps=6)["fp64"]
    assert s["steps_per_launch"] == plan
    assert s["roofline_frac"] == pytest.approx(n * n * 6 * 38 * 8 / (plan * 1e-3) / 8e12, abs=6e-5)


def test_a_single_step_is_a_launch_of_its_own(monkeypatch):
    monkeypatch.setattr(_Lattice, "plan", 2)
    r = bench.run_dense(_Module, np.zeros((16, 16, 16), bool), 16, 0.6, 0, 1, 1, 0.0)["roofline"]
    assert r["steps_per_launch"] == 1
