"""A handle's scratch under growth, capture and close, on the CPU: tests/native/arena_check.cpp links
the library's objects with a HIP runtime that has no device (device memory is host memory, kernels
are recorded and not run) and counts what the calls allocate, free and launch."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "rocket-userspace_amd")


def test_scratch_under_growth_and_capture(tmp_path):
    lib = os.path.join(PKG, "librocketnpu.a")
    src = os.path.join(REPO, "tests", "native", "arena_check.cpp")
    cxx = "/opt/rocm/llvm/bin/clang++"
    if not os.path.exists(cxx) or not os.path.exists(lib) or not os.path.exists(src):
        pytest.skip("needs clang++ and the static library")
    exe = str(tmp_path / "arena_check")
    b = subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(REPO, "include"), "-I", os.path.join(PKG, "csrc"),
                        "-I/opt/rocm/include", src, lib, "-o", exe,
                        "-lm", "-lpthread"], capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stdout[-3000:] + b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout[-2000:] + r.stderr[-4000:]
