"""The FFT building blocks of the transforms, run through their host paths
against a naive DFT: the Stockham stages (fft_core.hpp) at every length that
has no two-factor transform, both directions, and the two-factor transforms
(fft_reg.hpp) at every length, in FP32 also whether their error scales the
result.  CPU only; needs hipcc."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC) and shutil.which("hipcc") is None, reason="hipcc not available")
def test_fft_plans_against_naive_dft(tmp_path):
    exe = tmp_path / "fft_host_check"
    inc = os.path.join(os.path.dirname(HERE), "tinker-gpu_amd", "csrc")
    cc = HIPCC if os.path.exists(HIPCC) else "hipcc"
    subprocess.run([cc, "-std=c++17", "-O2", "-I", inc, os.path.join(HERE, "fft_host_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
