"""The host layer's C++ interface, through host_checks.cpp (no GPU needed)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("checks") / "host_checks")
    lib = os.path.join(ROOT, "glow_amd")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "include"),
                           os.path.join(ROOT, "tests", "host_checks.cpp"), "-o", exe, "-L" + lib,
                           "-lglow_mi355x_host", "-lglow_mi355x", "-Wl,-rpath," + lib,
                           "-Wl,-rpath-link,/opt/rocm/lib"])
    return exe


@pytest.mark.parametrize("check", ["bag_offsets", "downward", "upward", "flushed", "helpers_of_three_cpus"])
def test_check(checks, check):
    r = subprocess.run([checks, check], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
