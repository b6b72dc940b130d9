"""The large readouts (madpac_amd/csrc/lbm_readout.cpp) on the host, over a stand-in for the runtime
(tests/cpp/test_readout.cpp): pieces and threads, and what is left of them when memory runs out."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("readout") / "test_readout")
    csrc = os.path.join(ROOT, "madpac_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", csrc,
                    os.path.join(ROOT, "tests", "cpp", "test_readout.cpp"), os.path.join(csrc, "lbm_readout.cpp"),
                    "-o", out, "-pthread", "-ldl"], check=True)
    return out


def _run(*args):
    r = subprocess.run(args, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (args[1:], r.returncode, r.stdout, r.stderr)


def test_parts_arrive_whole(exe):
    _run(exe, "whole")


@pytest.mark.parametrize("started", [1, 3, 7])
def test_running_out_of_memory_between_threads(exe, started):
    # the threads that were started move every piece; the process goes on
    _run(exe, "nothreads", str(started))


def test_memory_that_the_runtime_knows_is_copied_to_directly(exe):
    _run(exe, "known")
