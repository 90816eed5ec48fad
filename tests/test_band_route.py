"""Which banded pairs the band kernel takes, at the limits of its int32 counts
and H (takes_band, anchorwave_amd/csrc/ksw2_batch.cpp): host only, through
tests/c/route_check.cpp linked to the library."""
import os
import shutil
import subprocess

import pytest

from anchorwave_amd import ksw2

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_band_domain(tmp_path):
    exe = tmp_path / "route_check"
    lib = os.path.dirname(ksw2.LIB_PATH)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "c", "route_check.cpp"), ksw2.LIB_PATH, f"-Wl,-rpath,{lib}",
                    "-Wl,--allow-shlib-undefined", "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "route ok" in r.stdout
