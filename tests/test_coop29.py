"""The point additions shared by groups of lanes (nkr-zkp_amd/csrc/coop29.h),
which the MSM bucket reduction is made of: their device code compiled for the
CPU, run on 16 emulated lanes with operands at the top of the bounds the
additions accept, through doublings, cancellations and infinity operands, and
compared with the canonical additions of curve.h."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_shared_additions_against_canonical_ones(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "coop29_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "nkr-zkp_amd", "csrc"), "-w",
                    os.path.join(ROOT, "tests", "host", "coop29_check.cpp"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    adds, doublings, cancels = [int(w) for w in res.stdout.replace("(", " ").split() if w.isdigit()]
    assert adds > 5000 and doublings > 300 and cancels > 300
