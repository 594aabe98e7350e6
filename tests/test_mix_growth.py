"""Host check (CPU) of how the error of the mixed-radix transforms grows over
the steps of an evolution, beside direct sums of table products."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_mixed_radix_errors_beside_direct_sums(tmp_path):
    exe = str(tmp_path / "mix_growth_check")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17",
           "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "qusim_amd", "csrc"),
           "-x", "hip", os.path.join(ROOT, "tests", "cpp", "mix_growth_check.cpp"), "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:]
    assert "error growth ok" in r.stdout
