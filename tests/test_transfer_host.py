"""The pinned ring and its helper threads (transfer.hpp) on the CPU, the runtime's calls replaced by host/hip."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "gaugefields.jl_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("transfer") / "transfer")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-pthread", "-I", os.path.join(HERE, "host"),
                    "-I", CSRC, os.path.join(HERE, "host", "transfer.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["failed_wait", "coherent", "late_helper", "blocked_signal",
                                      "small_transfer", "several_threads"])
def test_transfer(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
