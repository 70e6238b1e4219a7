"""The kept workspace of the stand-alone entry points when an allocation or a
copy fails, on the CPU: the library over a HIP runtime of host memory whose calls
can be made to fail (tests/cpp/fake_hip.c)."""
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT

PRELUDE = """
import ctypes, sys
import numpy as np
sys.path.insert(0, %r)
import ibpm_amd as gpu
fake = ctypes.CDLL(%r)
ctx = gpu.Context(0)
w = np.ones(31 * 31)
def solve(n=32):
    return ctx.elliptic2d_solve(0, n, n, 0.1, 0.0, np.ones((n - 1) * (n - 1)))
"""


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-Wall", os.path.join(ROOT, "tests", "cpp", "fake_hip.c"),
                    "-o", so], check=True)
    return so


def run(fake_hip, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE % (ROOT, fake_hip) + body], capture_output=True, text=True,
                       env=dict(os.environ, LD_PRELOAD=fake_hip), timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


def test_pinned_allocation_fails_then_succeeds(fake_hip):
    """The first descriptor upload finds no pinned memory: an error, and the
    next call is an ordinary one."""
    run(fake_hip, """
fake.fake_fail(b"hipHostMalloc", 0)
try:
    solve()
    raise SystemExit("no error")
except gpu.IbpmError as e:
    assert "out of memory" in str(e), e
assert fake.fake_failed()
solve()
solve()
""")


def test_workspace_that_cannot_grow_is_not_an_error(fake_hip):
    """A call that served itself by allocating succeeds although the workspace
    could not be kept, and leaves no error for the next one."""
    run(fake_hip, """
solve()
d = gpu.DeviceArray.of(ctx, np.ones(63 * 63)); u = gpu.DeviceArray(ctx, 63 * 63)
call = lambda: gpu.load().ibpm_elliptic2d_solve(ctx.h, 0, 64, 64, 0.1, 0.0, d.ptr, None, u.ptr)
# a 64 x 64 solve allocates scratch rows, boundary values and tables, then the larger workspace
for skip in range(8):
    ctx2 = gpu.Context(0)
    call2 = lambda: gpu.load().ibpm_elliptic2d_solve(ctx2.h, 0, 64, 64, 0.1, 0.0, d.ptr, None, u.ptr)
    fake.fake_fail(b"hipMalloc", skip)
    first = call2()
    if not fake.fake_failed():
        fake.fake_fail(b"none", 0)
    # whatever failed, and whether or not the call could do without it, the next is ordinary
    assert call2() == 0, (skip, first, gpu.load().ibpm_last_error())
    assert call2() == 0
    del ctx2
""")


def test_scope_that_ends_early_waits_for_its_work(fake_hip):
    """A copy fails after others were queued from the pinned descriptors: the
    call returns with the stream drained, as the next call reuses them."""
    run(fake_hip, """
n = 32
w = gpu.DeviceArray.of(ctx, np.ones(31 * 31)); q = gpu.DeviceArray(ctx, 2 * n * n + 2 * n)
call = lambda: gpu.load().ibpm_flux_from_vorticity(ctx.h, n, n, 1, 0.1, 0.0, 0.0, w.ptr, q.ptr)
assert call() == 0 and call() == 0
fake.fake_fail(b"hipMemcpyAsync", 1)   # the solve's descriptors go up, the curl's do not
assert call() != 0 and fake.fake_failed()
assert fake.fake_pending() == 0
assert call() == 0
""")
