"""One step of every model on multi-level grids of four cells a side, where the
nodes outside the corners of a coarse level's central region lie on the level's
boundary, against the FP64 CPU oracle."""
import numpy as np
import pytest

from tests.helpers import G

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4, 2), (4, 16, 2), (16, 4, 2), (4, 40, 2), (8, 4, 2),
          # fluxes of a central region that go down through the levels between
          (16, 4, 3), (4, 16, 3), (4, 4, 4), (4, 40, 5)]
MODELS = ["nonlinear", "linear", "adjoint", "sfd", "ubf"]


def case(nx, ny, model):
    h = 2.0 / nx   # the widest square that fits is one point at the centre
    mot = "  center 0 0\n  motion pitchplunge 0.3 0.4 0 0.1 0.3 0\n" if model == "ubf" else ""
    return "body P\n  point %.17g %.17g\n" % (0.1 * h, -0.2 * h) + mot + "end\n"


@pytest.mark.parametrize("model", MODELS)
@pytest.mark.parametrize("shape", SHAPES)
def test_one_step_on_the_smallest_levels(gpu, oracle, shape, model):
    nx, ny, L = shape
    print("smallest levels", shape, model, flush=True)
    g = G(nx, ny, L, 2.0, -1.0, -1.0 * ny / nx)
    geom = case(nx, ny, model)
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
