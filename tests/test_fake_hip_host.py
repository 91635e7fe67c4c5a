"""libpn1's host code on the CPU, over a HIP runtime of its own in host memory
(tests/fake_hip.hpp), which can refuse allocations, checks the arguments of every
launch and says how long launches took."""
import os
import shutil
import subprocess

import pytest

from pn_amd import build as b

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("name", ["ens_refused_check", "tuner_check"])
def test_over_fake_hip(tmp_path, name):
    """ens_refused_check: after a refused allocation an ensemble launches nothing
    of an earlier state or plan, and goes on.  tuner_check: the shape that is
    timed first, on a cold clock, is chosen if it is the fastest."""
    cc = shutil.which("g++")
    if cc is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("g++ or the HIP headers not available")
    if not os.path.exists(b.LIB):
        b.build()
    exe = str(tmp_path / name)
    subprocess.run([cc, "-O1", "-g", "-std=c++17", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                    "-I", b.INCLUDE, "-I", "/opt/rocm/include",
                    os.path.join(HERE, name + ".cpp"), b.LIB,
                    f"-Wl,-rpath,{b.HERE}", "-Wl,-rpath,/opt/rocm/lib", "-Wl,--allow-shlib-undefined",
                    "-o", exe], check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
