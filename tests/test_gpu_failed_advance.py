"""An advance that stops with an error after some of its steps: the flux is that
of the last completed step, as the vorticity and the forces are."""
import numpy as np
import pytest

from tests.helpers import plate_geom

pytestmark = pytest.mark.gpu

GRID = (64, 64, 2, 4.0, -2.0, -2.0, 100.0, 0.01)
FIXED = "body P\n line_n -0.5 0 0.5 0 9\n center 0 0\n motion fixed 0 0 -0.3\nend\n"
UBF = "body P\n line_n -0.5 0 0.5 0 9\n center 0 0\n motion pitchplunge 0.2 0.4 0 0.1 0.4 0\nend\n"
CASES = {"stationary": (FIXED, {}), "graph": (FIXED, {}), "adjoint": (FIXED, {"model": "adjoint"}),
         "moving": (plate_geom(9), {"tol": 1e-10}), "base flow": (UBF, {"ubf": True})}
LAST = (1 << 16) - 3   # three steps before the force history is full


@pytest.mark.parametrize("name", list(CASES))
def test_flux_after_an_advance_that_fails(gpu, name):
    geom, args = CASES[name]
    print("failed advance", name, flush=True)
    rng = np.random.default_rng(3)

    def batch():
        b = gpu.Batch(gpu.Context(0), [gpu.Flow(*GRID, geom, **args)])
        if args.get("model") == "adjoint":
            b.set_base_state(np.ones(2 * 63 * 63), np.full(2 * (2 * 64 * 64 + 128), 0.05))
        b.init()
        return b.use_graph(name == "graph")

    w = rng.standard_normal(2 * 63 * 63)
    a, c = batch(), batch()
    for b in (a, c):
        b.set_state(w, np.zeros(2 * b.num_points()), LAST * GRID[7], LAST)
    q0 = a.q()
    with pytest.raises(gpu.IbpmError, match="history capacity"):
        a.advance(5)
    c.advance(3)   # the steps that the history has room for
    assert np.array_equal(a.omega(), c.omega())
    assert np.array_equal(a.q(), c.q())
    assert not np.array_equal(a.q(), q0)
    with pytest.raises(gpu.IbpmError, match="history capacity"):   # no step at all: nothing changes
        a.advance(1)
    assert np.array_equal(a.q(), c.q())
