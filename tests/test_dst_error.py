"""Rounding error of the FP64 transforms of every compiled length, on the CPU:
no larger than that of the radix 8, 4, 2, 5, 3 transform they replaced."""
import os
import subprocess

from tests.conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_no_length_has_a_larger_error(tmp_path):
    exe = str(tmp_path / "dst_error_test")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O2", "-mavx2", "-mfma", "-ffp-contract=fast",
                    "-I", os.path.join(ROOT, "ibpm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "dst_error_test.cpp"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
