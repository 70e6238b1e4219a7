"""The DST passes at every transform length they are compiled for, along both
axes, against the FP64 CPU oracle: single levels with explicit boundary values,
multi-domain solves, and the rows of psi that the force solve reads when a
body lies next to the edge of the finest level."""
import numpy as np
import pytest

from tests.helpers import G

pytestmark = pytest.mark.gpu


def lengths():
    """Cells per side of every plan: 2..1024 with factors 2, 3, 5."""
    out = []
    for n in range(2, 1025):
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            out.append(n)
    return out


@pytest.fixture(scope="module")
def ctx(gpu):
    return gpu.Context(0)


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# Relative L2 of a solve: a few ulps times log2 of the transform lengths, as
# the multi-domain solves of the parity tests (1e-12).
@pytest.mark.parametrize("part", range(6))
def test_single_level_with_boundary_values(ctx, oracle, part):
    for n in lengths()[part::6]:
        for nx, ny, kind in ((n, 30, 0), (25, n, 1)):
            print("level", nx, ny, kind, flush=True)
            rng = np.random.default_rng(nx * 1025 + ny)
            f = rng.standard_normal((nx - 1) * (ny - 1))
            bc = rng.standard_normal(2 * (nx + ny))
            u = ctx.elliptic2d_solve(kind, nx, ny, 0.02, -1e-4, f, bc)
            assert rel(u, oracle.elliptic2d_solve(kind, nx, ny, 0.02, -1e-4, f, bc)) < 1e-12


@pytest.mark.parametrize("part", range(6))
def test_levels_couple_through_the_boundary_values(ctx, oracle, part):
    for n in [m for m in lengths() if m % 4 == 0][part::6]:
        for nx, ny, kind in ((n, 36, 1), (20, n, 0)):
            print("levels", nx, ny, kind, flush=True)
            f = np.random.default_rng(nx * 1025 + ny).standard_normal(3 * (nx - 1) * (ny - 1))
            u = ctx.elliptic_solve(kind, nx, ny, 3, 0.02, -1e-4, f)
            assert rel(u, oracle.elliptic_solve(kind, nx, ny, 3, 0.02, -1e-4, f)) < 1e-12


@pytest.mark.parametrize("cells", [1.7, 2.5, 4.5])
def test_body_next_to_the_edge_of_the_finest_level(gpu, ctx, oracle, cells):
    n, dx = 64, 4.0 / 64
    x = -2 + cells * dx
    geom = "body P\n" + "".join("  point %.17g %.17g\n" % (x, y) for y in np.linspace(-0.3, 0.3, 9))
    geom += "  center %.17g 0\n  motion pitchplunge 0.02 0.3 0 0.05 0.3 0\nend\n" % x
    b = gpu.Batch(ctx, [gpu.Flow(n, n, 2, 4.0, -2.0, -2.0, 100.0, 0.01, geom, tol=1e-10)]).init()
    s = oracle.Sim(n, n, 2, 4.0, -2.0, -2.0, 100.0, 0.01, geom, tol=1e-10)
    s.init()
    b.advance(2)
    s.advance(2)
    assert rel(b.omega(), s.omega()) < 1e-7
    assert rel(b.f(), s.f()) < 1e-6   # the CG tolerance's effect on the point forces
