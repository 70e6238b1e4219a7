"""Interpolation to and smearing from body points where their lists change
shape: component counts about one block's groups, slots touched by one or many
points, bodies within reach of the domain's edge, against the FP64 CPU oracle."""
import numpy as np
import pytest

from tests.helpers import G

pytestmark = pytest.mark.gpu

# name: (columns, rows of points, spacing in cells, first point's cell offset)
BODIES = {
    "one": (1, 1, 1.0, (16.3, 16.4)),
    "line7": (7, 1, 1.5, (9.2, 16.1)),          # 14 components, under one block's 16 groups
    "line9": (9, 1, 1.5, (9.2, 16.1)),          # 18, past it
    "rows": (9, 2, 1.2, (9.2, 16.1)),           # up to six entries in a slot; cond(M) = 3e2
    "edge": (3, 2, 2.0, (2.6, 2.7)),            # lists with fluxes beside the level's edge
}


def geometry(g, cols, rows, h, offset):
    ox, oy = offset
    pts = "".join("  point %.17g %.17g\n" % (-1 + g.dx * (ox + h * i), -1 + g.dx * (oy + h * j))
                  for i in range(cols) for j in range(rows))
    return "body P\n" + pts + "end\n"


@pytest.mark.parametrize("levels", [1, 3])
@pytest.mark.parametrize("name", sorted(BODIES))
def test_step_with_body(gpu, oracle, name, levels):
    cols, rows, h, offset = BODIES[name]
    print("body lists", name, levels, flush=True)
    n = 32
    g = G(n, n, levels, 2.0, -1.0, -1.0)
    geom = geometry(g, cols, rows, h, offset)
    args = dict(scheme="rk3", model="nonlinear")
    b = gpu.Batch(gpu.Context(0), [gpu.Flow(n, n, levels, 2.0, -1.0, -1.0, 80.0, 0.004, geom, **args)])
    s = oracle.Sim(n, n, levels, 2.0, -1.0, -1.0, 80.0, 0.004, geom, **args)
    b.init()
    s.init()
    w = np.random.default_rng(cols + rows).standard_normal(levels * g.ns)
    b.set_omega(w)
    s.set_omega(w)
    b.advance(2)
    s.advance(2)
    # a few ulps per operation times the force solve's conditioning (below 1e4)
    assert np.linalg.norm(b.omega() - s.omega()) <= 1e-10 * np.linalg.norm(s.omega())
    assert np.linalg.norm(b.q() - s.q()) <= 1e-10 * np.linalg.norm(s.q())


@pytest.mark.parametrize("levels", [1, 3])
def test_a_filled_patch_is_refused(gpu, levels):
    """A 5 x 5 patch of points has a force that smears to a curl-free field: M's
    smallest eigenvalue is 7e-20 against 1e-3, and the oracle, which does not
    look at its pivots, runs into NaN."""
    g = G(32, 32, levels, 2.0, -1.0, -1.0)
    geom = geometry(g, 5, 5, 1.3, (12.1, 12.2))
    b = gpu.Batch(gpu.Context(0), [gpu.Flow(32, 32, levels, 2.0, -1.0, -1.0, 80.0, 0.004, geom,
                                            scheme="rk3", model="nonlinear")])
    with pytest.raises(gpu.IbpmError, match="not positive definite"):
        b.init()
