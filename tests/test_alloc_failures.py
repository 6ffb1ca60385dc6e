"""Allocations that fail, each in turn, on the CPU: tests/alloc_failures.cpp
over the built library and a stand-in for the HIP runtime."""
import os
import subprocess

import pytest

import phylommand_amd as P

HERE = os.path.dirname(os.path.abspath(__file__))


def test_no_launch_without_its_memory(tmp_path):
    if not os.path.exists(P.LIB_PATH):
        pytest.skip("library not built")
    lib_dir = os.path.dirname(P.LIB_PATH)
    exe = str(tmp_path / "alloc_failures")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-rdynamic", "-o", exe,
                           os.path.join(HERE, "alloc_failures.cpp"), "-L" + lib_dir, "-lphylo_hip",
                           "-Wl,-rpath," + lib_dir, "-Wl,--allow-shlib-undefined"])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.startswith("ok"), (out.stdout + out.stderr)[:4000]
