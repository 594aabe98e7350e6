"""Host check (CPU) of the twiddle powers that the 1D lines hold in registers."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_twiddle_powers_are_no_further_off_than_the_recurrence(tmp_path):
    exe = str(tmp_path / "twiddle_powers_check")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17",
           "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "qusim_amd", "csrc"),
           "-x", "hip", os.path.join(ROOT, "tests", "cpp", "twiddle_powers_check.cpp"), "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:]
    assert "twiddle powers ok" in r.stdout
