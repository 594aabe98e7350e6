"""Host check (CPU) of the mixed-radix plans (qsim_mix.h): the set of lengths
they take, radices, pass indexes, twiddle indexes, launch shapes, and the
values of the kernels' own butterflies against a long double DFT."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_mixed_radix_plans_against_a_long_double_dft(tmp_path):
    exe = str(tmp_path / "mix_check")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17",
           "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "qusim_amd", "csrc"),
           "-x", "hip", os.path.join(ROOT, "tests", "cpp", "mix_check.cpp"), "-o", exe]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:]
    assert "mixed plans ok" in r.stdout
