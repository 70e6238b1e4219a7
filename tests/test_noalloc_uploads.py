"""The allocation-free solve uploads its tables and descriptors in one copy, and
accepts every grid that fits its array.  On the CPU, over a HIP runtime of host
memory (tests/cpp/fake_hip.c)."""
import os
import subprocess
import sys

from tests.conftest import ROOT

BODY = """
import ctypes, sys
import numpy as np
sys.path.insert(0, %r)
import ibpm_amd as gpu
fake = ctypes.CDLL(%r)
ctx = gpu.Context(0)
d = gpu.DeviceArray(ctx, 8 << 20); u = gpu.DeviceArray(ctx, 8 << 20)
def call(nx, ny, L):
    fake.fake_uploads()
    return gpu.load().ibpm_elliptic_solve_noalloc(ctx.h, 0, nx, ny, L, 0.1, 0.0, d.ptr, u.ptr)
for grid in ((64, 64, 1), (3, 5, 1), (225, 150, 1), (4, 4, 16), (400, 400, 4), (512, 512, 5), (1024, 64, 3),
             (960, 960, 1), (1024, 4, 16)):
    assert call(*grid) == 0, (grid, gpu.load().ibpm_last_error())
    assert fake.fake_uploads() == 1, grid
assert call(1024, 1024, 2) == -2 and call(64, 64, 17) == -2
assert fake.fake_uploads() == 0
"""


def test_one_upload_per_call(tmp_path):
    so = str(tmp_path / "fake_hip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", os.path.join(ROOT, "tests", "cpp", "fake_hip.c"), "-o", so],
                   check=True)
    r = subprocess.run([sys.executable, "-c", BODY % (ROOT, so)], capture_output=True, text=True,
                       env=dict(os.environ, LD_PRELOAD=so), timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
