"""Idle work blocks (sonium_amd/csrc/work_pool.cpp) on the host: limits for
device and pinned memory, reuse, allocations of either kind that find the memory
full of idle blocks, and threads that exchange blocks, against a model of the
runtime's allocation calls (tests/host/work_pool_driver.cpp)."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_idle_blocks_against_a_model_of_the_runtime(tmp_path):
    exe = tmp_path / "work_pool"
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "sonium_amd", "csrc"),
           os.path.join(ROOT, "sonium_amd", "csrc", "work_pool.cpp"),
           os.path.join(ROOT, "tests", "host", "work_pool_driver.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
