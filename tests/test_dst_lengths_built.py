"""Transform lengths that the plans accept and those that are compiled
(dst_f64.hip): the same set, and a plan of a length that is not compiled is
refused (its launches would do nothing).  On the CPU, over a HIP runtime of host
memory (tests/cpp/fake_hip.c)."""
import os
import subprocess
import sys

from tests.conftest import ROOT

BODY = """
import sys
import numpy as np
sys.path.insert(0, %r)
import ibpm_amd as gpu
ctx = gpu.Context(0)
def smooth(n):
    for p in (2, 3, 5):
        while n %% p == 0:
            n //= p
    return n == 1
def accepted(n):
    d = gpu.DeviceArray(ctx, 3 * (n - 1)); u = gpu.DeviceArray(ctx, 3 * (n - 1))
    return gpu.load().ibpm_elliptic2d_solve(ctx.h, 0, n, 4, 0.1, 0.0, d.ptr, None, u.ptr) == 0
"""


def run(tmp_path, body, missing=0):
    so = str(tmp_path / "fake_hip.so")
    src = [os.path.join(ROOT, "tests", "cpp", "fake_hip.c")]
    if missing:   # the library's own answer replaced: one length is not compiled
        stub = tmp_path / "missing.c"
        stub.write_text("_Bool _ZN5ibpmg16dst_length_builtEi(int m) { return m != %d; }\n" % missing)
        src.append(str(stub))
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1"] + src + ["-o", so], check=True)
    r = subprocess.run([sys.executable, "-c", BODY % ROOT + body], capture_output=True, text=True,
                       env=dict(os.environ, LD_PRELOAD=so), timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


def test_every_accepted_length_is_compiled(tmp_path):
    run(tmp_path, """
ok = [n for n in range(2, 1040) if accepted(n)]
assert ok == [n for n in range(2, 1025) if smooth(n)], ok
assert len(ok) == 86
""")


def test_a_length_that_is_not_compiled_is_refused(tmp_path):
    run(tmp_path, """
assert accepted(64) and not accepted(60)
assert b"no transform of length 120" in gpu.load().ibpm_last_error()
""", missing=120)
