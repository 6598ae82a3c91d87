"""Launch and index arithmetic for up to 2^32 - 1 items (a photon grid is
accepted up to that many cells): tests/cpu/count_check.cpp, built with hipcc
here and run on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "differentiablepointrendering_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None, reason="needs hipcc")
def test_counts(tmp_path):
    exe = str(tmp_path / "count_check")
    cc = HIPCC if os.path.exists(HIPCC) else "hipcc"
    subprocess.run([cc, "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "cpu", "count_check.cpp"), "-o", exe], check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
