"""Host check (CPU) of the lengths that the mixed-radix lines leave to the
generic kernel and the unfused order: a refused plan is empty, the refused set
is what the LDS arithmetic gives, and the lengths of test_gpu_handover.py are
in it."""
import os
import shutil
import subprocess

import pytest

from test_gpu_handover import REFUSED

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_refused_mixed_radix_plans_are_empty(tmp_path):
    exe = str(tmp_path / "mix_refused_check")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17",
           "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "qusim_amd", "csrc"),
           "-x", "hip", os.path.join(ROOT, "tests", "cpp", "mix_refused_check.cpp"), "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([exe] + [str(n) for n in REFUSED], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout[-2000:]
    assert "refused plans ok" in r.stdout
