"""Stand-alone entry points on one context's kept workspace: calls of changing
sizes, outputs that alias or overlap their inputs, and two contexts driven from
two threads give bit for bit what fresh contexts give."""
import threading

import numpy as np
import pytest

from tests.helpers import G

pytestmark = pytest.mark.gpu

# sizes around the workspace's growth: small, larger, back, several levels
GRIDS = [(16, 24, 1), (64, 48, 3), (12, 20, 2), (200, 160, 2), (64, 48, 3)]


def call_all(ctx, nx, ny, L):
    g = G(nx, ny, L, 2.0, -1.0, -1.0)
    rng = np.random.default_rng(nx * L)
    w, n = rng.standard_normal(L * g.ns), rng.standard_normal(L * g.ns)
    q = rng.standard_normal(L * g.nf)
    a = (nx, ny, L, g.dx)
    out = [ctx.elliptic_solve(0, *a, 0.0, w), ctx.elliptic_solve(1, *a, -1e-4, w), ctx.curl_flux(*a, q),
           ctx.laplacian(*a, w), ctx.curl_scalar(*a, w, 1.0, 0.5), ctx.nonlinear(*a, q, w), ctx.cross_product(*a, q, w),
           ctx.cross_flux_flux(*a, q, q[::-1].copy()), ctx.flux_from_vorticity(*a, w, 1.0, 0.5)]
    return out + list(ctx.rhs(*a, 0.01, 0.02, 5 / 12, -17 / 60, q, w, n)) + [ctx.dst2d(w[:g.ns].reshape(nx - 1, ny - 1))]


def test_kept_workspace_equals_fresh_contexts(gpu):
    ctx = gpu.Context(0)
    for grid in GRIDS:
        print("workspace", grid, flush=True)
        for a, b in zip(call_all(ctx, *grid), call_all(gpu.Context(0), *grid)):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("shift", [0, 7, -7])
def test_solution_over_its_right_hand_side(gpu, shift):
    ctx = gpu.Context(0)
    nx, ny, L = 32, 40, 3
    ns = (nx - 1) * (ny - 1)
    f = np.random.default_rng(3).standard_normal(L * ns)
    want = ctx.elliptic_solve(0, nx, ny, L, 0.1, 0.0, f)
    buf = np.zeros(L * ns + 16)
    buf[8:8 + L * ns] = f
    d = gpu.DeviceArray.of(ctx, buf)
    print("overlap", shift, flush=True)
    rc = gpu.load().ibpm_elliptic_solve(ctx.h, 0, nx, ny, L, 0.1, 0.0, d.ptr.value + 64, d.ptr.value + 64 + 8 * shift)
    assert rc == 0 and np.array_equal(d.get()[8 + shift:8 + shift + L * ns], want)


def test_two_contexts_on_two_threads(gpu):
    want = [call_all(gpu.Context(0), *g) for g in GRIDS]
    bad = []

    def work(order):
        try:
            ctx = gpu.Context(0)
            for k in order:
                bad.extend(k for a, b in zip(call_all(ctx, *GRIDS[k]), want[k]) if not np.array_equal(a, b))
        except Exception as e:   # reported after the join
            bad.append(e)
    th = [threading.Thread(target=work, args=(o,)) for o in ([0, 1, 2, 3, 4], [3, 0, 4, 1, 2])]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
