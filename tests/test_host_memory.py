"""Shortage of device memory: at every allocation of an operation the call
reports it, a second call on the same graph does too (it does not go on with
what the first one left), a call with memory again works, and nothing is lost.
Rows in managed memory: not for a kernel that lowers distances in them.
The library's host code runs on stand-ins for the HIP runtime
(tests/host_hip.cpp); no GPU."""
import os
import subprocess

import pytest

from conftest import ROOT

PKG = os.path.join(ROOT, "gal-dawn_amd")
OPERATIONS = ("bfs", "sssp", "weighted_lanes_8", "weighted_lanes_64", "weighted_workgroups", "lanes",
              "lanes_hub_order", "workgroups", "workgroups_no_rows", "batch", "batch_weighted")


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_hip") / "host_hip")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"),
                    "-I", "/opt/rocm/include", os.path.join(ROOT, "tests", "host_hip.cpp"), "-o", exe,
                    "-L", PKG, "-ldawn_amd", f"-Wl,-rpath,{PKG}", "-Wl,-rpath,/opt/rocm/lib",
                    "-Wl,-rpath-link,/opt/rocm/lib"], check=True)
    return exe


def test_operations_listed(host_hip):
    assert set(subprocess.run([host_hip, "list"], capture_output=True, text=True).stdout.split()) == set(OPERATIONS)


@pytest.mark.parametrize("operation", OPERATIONS)
def test_memory_shortage(host_hip, operation):
    r = subprocess.run([host_hip, "memory", operation], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_managed_rows(host_hip):
    r = subprocess.run([host_hip, "managed"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
