"""A captured step of flows of different transform lengths, whose solves are
branches of the graph: every replay equals the step launched on one stream, bit
for bit (the kernels are the same), with two lengths, more lengths than
branches, and levels that only some of the flows have."""
import numpy as np
import pytest

from tests.helpers import G

pytestmark = pytest.mark.gpu

BATCHES = {
    "two lengths": [(64, 64, 3), (96, 96, 3), (64, 64, 3)],
    "six lengths": [(32, 32, 2), (64, 64, 1), (48, 32, 3), (96, 64, 2), (80, 80, 4), (128, 128, 2), (64, 64, 3)],
    "one level": [(50, 40, 1), (64, 64, 1), (40, 50, 1)],
}


@pytest.mark.parametrize("name", sorted(BATCHES))
def test_replays_equal_one_stream(gpu, name):
    print("branches", name, flush=True)
    fl, start = [], []
    for k, (nx, ny, levels) in enumerate(BATCHES[name]):
        g = G(nx, ny, levels, 2.0, -1.0, -1.0 * ny / nx)
        h = 2.2 * g.dx
        pts = "".join("  point %.17g %.17g\n" % p for p in ((-h, -h), (h, -h), (-h, h), (h, h)))
        fl.append(gpu.Flow(nx, ny, levels, 2.0, -1.0, -1.0 * ny / nx, 80.0 + k, 0.004,
                           "body P\n" + pts + "end\n", scheme="rk3", model="nonlinear"))
        start.append(np.random.default_rng(k).standard_normal(levels * g.ns))
    ctx = gpu.Context(0)
    graph = gpu.Batch(ctx, fl).init()
    plain = gpu.Batch(ctx, fl).init()
    plain.use_graph(False)
    for b in (graph, plain):
        for k, w in enumerate(start):
            b.set_omega(w, k)
    for step in range(6):   # the first runs before the step is captured
        graph.advance(1)
        plain.advance(1)
        for k in range(len(fl)):
            assert np.array_equal(graph.omega(k), plain.omega(k)), (step, k)
            assert np.array_equal(graph.q(k), plain.q(k)), (step, k)
            assert np.array_equal(graph.f(k), plain.f(k)), (step, k)
