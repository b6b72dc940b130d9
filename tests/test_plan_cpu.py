"""Planning the launches of a run of steps, on the host."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "test_plan")
    lib = os.path.join(ROOT, "madpac_amd")
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(lib, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_plan.cpp"), "-o", exe, "-L" + lib, "-llbm_hip",
                    "-Wl,-rpath," + lib], check=True)

    def run(*args):
        r = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
        return r.stdout
    return run


def test_a_plan_costs_a_call_next_to_nothing(plan):
    # the search over chunk counts (up to 19 us on these lattices) belongs to the context, not to each call;
    # what is left is a few dozen operations: 2 us leave room for a slow host
    assert float(plan("cost")) < 2.0


@pytest.mark.parametrize("size, solids, esize, f32math, pairs", [
    # measured single / in pairs, us a step (table at pair_plan); force or porosity
    ((192, 192, 96), 0.1, 4, False, False),   # 100.3 / 105.8
    ((192, 192, 96), 0.0, 4, False, False),   # 94.4 / 100.0
    ((224, 200, 150), 0.1, 4, False, False),  # 219 / 232
    ((192, 192, 192), 0.1, 4, False, False),  # 195 / 204
    ((1000, 1000, 2), 0.1, 8, False, False),  # 130 / 138
    ((192, 192, 96), 0.1, 4, True, True),     # 102.1 / 100.0
    ((128, 128, 128), 0.1, 4, False, True),   # 60.7 / 56.5
    ((240, 240, 240), 0.1, 4, False, True),   # 472 / 416
    ((1000, 1000, 2), 0.0, 8, False, True),   # 120 / 92
    ((131, 70, 53), 0.1, 8, False, True),     # 36.8 / 32.8
])
def test_pairs_are_chosen_where_they_measured_faster(plan, size, solids, esize, f32math, pairs):
    cells = size[0] * size[1] * size[2]
    assert plan(*size, esize, int(f32math), int(cells * (1 - solids)), 1, 0, 0).strip() == str(int(pairs))
