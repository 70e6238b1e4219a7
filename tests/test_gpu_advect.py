"""A batch's stencils (N and the right-hand side formed straight from psi) at the
edges of their tiles and on the smallest grids, every model, against the FP64
CPU oracle: one Euler step and one RK3 step from a random vorticity."""
import numpy as np
import pytest

from tests.helpers import G

pytestmark = pytest.mark.gpu

# rows and columns below, at and past the 8 x 64 tiles; the coarse levels' rims
# inside one tile and across several
SHAPES = [(12, 16, 3), (20, 64, 2), (8, 72, 2), (72, 144, 3), (9, 75, 1), (36, 128, 4)]
MODELS = ["nonlinear", "linear", "adjoint", "sfd", "ubf"]


@pytest.mark.parametrize("model", MODELS)
@pytest.mark.parametrize("shape", SHAPES)
def test_one_step_from_random_vorticity(gpu, oracle, shape, model):
    nx, ny, L = shape
    print("advect", shape, model, flush=True)
    g = G(nx, ny, L, 2.0, -1.0, -1.0 * ny / nx)
    h = 2.2 * g.dx   # four points further apart than the regulariser's reach
    pts = "".join("  point %.17g %.17g\n" % p for p in ((-h, -h), (h, -h), (-h, h), (h, h)))
    mot = "  center 0 0\n  motion pitchplunge 0.3 0.4 0 0.1 0.3 0\n" if model == "ubf" else ""
    geom = "body P\n" + pts + mot + "end\n"
    name = "nonlinear" if model == "ubf" else model
    rng = np.random.default_rng(nx * ny + L)
    w0, q0 = rng.standard_normal(L * g.ns), g.dx * rng.standard_normal(L * g.nf)
    for scheme in ("euler", "rk3"):
        args = dict(scheme=scheme, model=name, ubf=model == "ubf")
        b = gpu.Batch(gpu.Context(0), [gpu.Flow(nx, ny, L, 2.0, -1.0, -1.0 * ny / nx, 80.0, 0.004, geom, **args)])
        s = oracle.Sim(nx, ny, L, 2.0, -1.0, -1.0 * ny / nx, 80.0, 0.004, geom, **args)
        if name in ("linear", "adjoint"):
            b.set_base_state(w0, q0)
            s.set_base_state(w0, q0)
        b.init()
        s.init()
        w = np.random.default_rng(5).standard_normal(L * g.ns)
        b.set_omega(w)
        s.set_omega(w)
        b.advance(1)
        s.advance(1)
        # a few ulps per operation, the force solve's conditioning (below 1e4) on top
        assert np.linalg.norm(b.omega() - s.omega()) <= 1e-11 * np.linalg.norm(s.omega())
        assert np.linalg.norm(b.q() - s.q()) <= 1e-11 * np.linalg.norm(s.q())
