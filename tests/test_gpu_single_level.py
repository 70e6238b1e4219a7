"""Stationary bodies on one level, where a substep's solves run in pairs from
one forward transform, against the FP64 CPU oracle: one-stage and odd lengths,
lengths that differ along i and j, an odd pair at either end, every model, and
a batch of several lengths."""
import numpy as np
import pytest

from tests.helpers import G

pytestmark = pytest.mark.gpu

SHAPES = [(12, 16), (16, 12), (20, 24), (45, 27), (64, 64), (75, 50), (200, 120)]


def body(g):
    h = 2.2 * g.dx   # four points further apart than the regulariser's reach
    pts = "".join("  point %.17g %.17g\n" % p for p in ((-h, -h), (h, -h), (-h, h), (h, h)))
    return "body P\n" + pts + "end\n"


def compare(b, s, k):
    # a few ulps per operation, the force solve's conditioning (below 1e4) on top
    assert np.linalg.norm(b.omega(k) - s.omega()) <= 1e-11 * np.linalg.norm(s.omega())
    assert np.linalg.norm(b.q(k) - s.q()) <= 1e-11 * np.linalg.norm(s.q())
    assert np.linalg.norm(b.f(k) - s.f()) <= 1e-9 * np.linalg.norm(s.f())


def pair(gpu, oracle, shapes, model, scheme):
    fl, sims, start = [], [], []
    for nx, ny in shapes:
        g = G(nx, ny, 1, 2.0, -1.0, -1.0 * ny / nx)
        a = (nx, ny, 1, 2.0, -1.0, -1.0 * ny / nx, 80.0, 0.004, body(g))
        fl.append(gpu.Flow(*a, scheme=scheme, model=model))
        sims.append(oracle.Sim(*a, scheme=scheme, model=model))
        rng = np.random.default_rng(nx * ny)
        start.append((rng.standard_normal(g.ns), g.dx * rng.standard_normal(g.nf), rng.standard_normal(g.ns)))
    b = gpu.Batch(gpu.Context(0), fl)
    for k, (w0, q0, _) in enumerate(start):
        if model in ("linear", "adjoint"):
            b.set_base_state(w0, q0, k=k)
            sims[k].set_base_state(w0, q0)
    b.init()
    for k, (_, _, w) in enumerate(start):
        sims[k].init()
        b.set_omega(w, k)
        sims[k].set_omega(w)
    return b, sims


@pytest.mark.parametrize("model", ["nonlinear", "adjoint", "sfd"])
@pytest.mark.parametrize("shape", SHAPES)
def test_steps_of_one_level(gpu, oracle, shape, model):
    for scheme in ("euler", "rk3"):
        print("single level", shape, model, scheme, flush=True)
        b, sims = pair(gpu, oracle, [shape], model, scheme)
        b.advance(3)
        sims[0].advance(3)
        compare(b, sims[0], 0)


def test_batch_of_several_lengths(gpu, oracle):
    shapes = [(20, 24), (64, 64), (24, 20), (64, 64)]
    print("single level batch", flush=True)
    b, sims = pair(gpu, oracle, shapes, "nonlinear", "rk3")
    b.advance(3)
    for k, s in enumerate(sims):
        s.advance(3)
        compare(b, s, k)
