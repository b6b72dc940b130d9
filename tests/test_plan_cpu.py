"""Planning the launches of a run of steps, on the host."""
import os
import subprocess

from conftest import ROOT


def test_a_plan_costs_a_call_next_to_nothing(tmp_path):
    # the search over chunk counts (up to 19 us on these lattices) belongs to the context, not to each call;
    # what is left is a few dozen operations: 2 us leave room for a slow host
    exe = str(tmp_path / "test_plan")
    lib = os.path.join(ROOT, "madpac_amd")
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(lib, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_plan.cpp"), "-o", exe, "-L" + lib, "-llbm_hip",
                    "-Wl,-rpath," + lib], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    assert float(r.stdout) < 2.0
