"""Refused allocations of an ensemble, on the CPU: tests/ens_refused_check.cpp
puts a HIP runtime of its own over host memory under libpn1.so, refuses each
allocation of a plan change, an upload and the tuner in turn, and checks the
arguments of every launch that follows (live buffers, work items of the
present state)."""
import os
import shutil
import subprocess

import pytest

from pn_amd import build as b

HERE = os.path.dirname(os.path.abspath(__file__))


def test_refused_allocations(tmp_path):
    cc = shutil.which("g++")
    if cc is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("g++ or the HIP headers not available")
    if not os.path.exists(b.LIB):
        b.build()
    exe = str(tmp_path / "ens_refused_check")
    subprocess.run([cc, "-O1", "-g", "-std=c++17", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                    "-I", b.INCLUDE, "-I", "/opt/rocm/include",
                    os.path.join(HERE, "ens_refused_check.cpp"), b.LIB,
                    f"-Wl,-rpath,{b.HERE}", "-Wl,-rpath,/opt/rocm/lib", "-Wl,--allow-shlib-undefined",
                    "-o", exe], check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.startswith("ok "), r.stdout + r.stderr
