"""Compiles a C++ test program with host sources of the library and the stand-in runtime, and runs it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ls-stag-3d_parallel_amd", "csrc")


def run(tmp_path, program, sources=()):
    cxx = next((c for c in ("/opt/rocm/llvm/bin/clang++", shutil.which("amdclang++")) if c and os.path.exists(c)), None)
    if cxx is None:
        pytest.skip("no clang++ of a ROCm installation")
    src, exe = tmp_path / "main.cpp", tmp_path / "main"
    src.write_text(program)
    # what a program does not call stays unresolved
    cmd = [cxx, "-x", "c++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           "-I", os.path.join(ROOT, "tests"), "-I", CSRC, "-no-pie", "-Wno-unused-result", str(src)]
    cmd += [os.path.join(CSRC, s) for s in sources] + ["-Wl,--unresolved-symbols=ignore-all", "-lpthread", "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr)
