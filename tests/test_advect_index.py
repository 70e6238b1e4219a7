"""Offsets of a batch's stencils on every small multi-level grid, checked on the
CPU: the index rules of advect.h, which the kernels use, compiled for the host."""
import os
import subprocess

from tests.conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_every_offset_is_inside_its_field(tmp_path):
    exe = str(tmp_path / "advect_index_test")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                    "-I", os.path.join(ROOT, "ibpm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "advect_index_test.cpp"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
