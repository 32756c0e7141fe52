"""Copies between host arrays and the device (nimbus_amd/csrc/host_transfer.hpp)
compiled for the host against a runtime interface on host memory
(tests/native/hip_on_host): which route a call takes, and that its arrays
arrive whole."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_transfer") / "check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I" + os.path.join(NATIVE, "hip_on_host"),
                        "-I" + os.path.join(ROOT, "nimbus_amd", "csrc"),
                        os.path.join(NATIVE, "host_transfer_check.cpp"), "-o", exe, "-pthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("check", ["small", "large", "reach", "foreign", "no_threads", "pinned", "no_memory", "shared"])
def test_host_transfer(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
