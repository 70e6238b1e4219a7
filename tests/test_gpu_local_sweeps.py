"""The local Helmholtz sweeps where their launches end: the largest substep's
sweep count below, at and past one launch's and two launches' worth, and boxes
of one tile and of several, against the DST solve of the same system."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT, DX = 0.005, 4.0 / 128


def sweeps(Re):
    """The sweep count of the substep with the largest beta = 8/15 dt on level 0."""
    c = 8.0 / 15.0 * DT / (2.0 * Re * DX * DX)
    return math.ceil(math.log(1e-18) / math.log(4 * c / (1 + 4 * c)))


def reynolds(count):
    """The middle of the Reynolds numbers that take `count` sweeps."""
    got = [Re for Re in np.geomspace(3.0, 3000.0, 4000) if sweeps(Re) == count]
    return float(got[len(got) // 2])


@pytest.mark.parametrize("points", [5, 65])
@pytest.mark.parametrize("count", [7, 12, 13, 24, 25])
def test_sweeps_equal_the_dst_solve(gpu, count, points):
    Re, half = reynolds(count), 0.5 * (points - 1) * DX / 2
    print("local sweeps", count, points, Re, flush=True)
    geom = ("body Plate\n  line_n %.17g 0.01 %.17g 0.01 %d\n  center 0 0\n"
            "  motion pitchplunge 0.2 0.4 0 0.2 0.4 0\nend\n" % (-half, half, (points + 1) // 2))
    ctx = gpu.Context(0)
    fl = gpu.Flow(128, 128, 3, 4.0, -2.0, -2.0, Re, DT, geom, tol=1e-10)
    loc = gpu.Batch(ctx, [fl]).init()
    dst = gpu.Batch(ctx, [fl]).init().set_local_helmholtz(False)
    loc.advance(3)
    dst.advance(3)
    sl = loc.solver_stats()
    assert sl["local_helmholtz_m_applications"] == sl["m_applications"] > 0
    # the conjugate gradients stop at 1e-10; its effect on forces and vorticity
    hl, hd = loc.force_history(), dst.force_history()
    assert np.abs(hl - hd).max() <= 1e-8 * np.abs(hd).max()
    assert np.linalg.norm(loc.omega() - dst.omega()) <= 1e-8 * np.linalg.norm(dst.omega())


@pytest.mark.parametrize("levels", [2, 4])
@pytest.mark.parametrize("reach", [20, 45, 58])
def test_coarse_right_hand_sides(gpu, reach, levels):
    """A diagonal plate of 2 reach cells: both coarsify chains within one
    workgroup's 3136 points on level 1 (reach 20), only the sweeps' own (45),
    neither (58); two flows, so that the second one's jobs do not start at 0."""
    n, dx, Re = 256, 8.0 / 256, 196.0
    print("coarse right-hand sides", reach, levels, flush=True)
    a, pts = reach * dx, reach + 1
    geom = ("body Plate\n  line_n %.17g %.17g %.17g %.17g %d\n  center 0 0\n"
            "  motion pitchplunge 0.1 0.4 0 0.1 0.4 0\nend\n" % (-a, -a + 0.01, a, a + 0.01, pts))
    small = ("body Plate\n  line_n -0.3 0.01 0.3 0.01 11\n  center 0 0\n"
             "  motion pitchplunge 0.1 0.4 0 0.1 0.4 0\nend\n")
    ctx = gpu.Context(0)
    fl = [gpu.Flow(n, n, levels, 8.0, -4.0, -4.0, Re, DT, g, tol=1e-10) for g in (small, geom)]
    loc = gpu.Batch(ctx, fl).init()
    dst = gpu.Batch(ctx, fl).init().set_local_helmholtz(False)
    loc.advance(2)
    dst.advance(2)
    sl = loc.solver_stats()
    assert sl["local_helmholtz_m_applications"] == sl["m_applications"] > 0
    for k in range(2):
        hl, hd = loc.force_history(k), dst.force_history(k)
        assert np.abs(hl - hd).max() <= 1e-8 * np.abs(hd).max()
        assert np.linalg.norm(loc.omega(k) - dst.omega(k)) <= 1e-8 * np.linalg.norm(dst.omega(k))
