"""The quotient by a density in hand (hx::quot, csrc/physics.hpp) has the bits of the division over the values
that a regular state has, and its exceptions are those it states (tests/host/quotient.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "horses3d_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_quotient_has_the_bits_of_the_division(tmp_path):
    if shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "include", "hip")):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "quotient")
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                        "-I", CSRC, os.path.join(HERE, "host", "quotient.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe, "4000000"], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
