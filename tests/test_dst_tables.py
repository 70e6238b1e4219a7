"""Tables of the transform plans on the CPU, against extended precision: every
twiddle, eigenvalue cosine and ring sine rounded to the nearest double (sines of
arguments up to 800 had lost three digits)."""
import os
import subprocess

from tests.conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_tables_are_rounded_from_extended_precision(tmp_path):
    exe = str(tmp_path / "dst_tables_test")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                    "-I", os.path.join(ROOT, "ibpm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "dst_tables_test.cpp"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
