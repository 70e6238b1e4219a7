"""Performance cases of the projection-step library: what a user of ibpm_amd has it do, from one small
elliptic solve to the batch of sixteen tandem-plate flows, each run through the public entry points.

Two kinds of call are covered:
- the operators of the C ABI on device arrays (a driver that keeps its own time loop): the multi-domain
  Poisson and Helmholtz solves, the flux of a vorticity field, the right-hand side of a substep;
- whole timesteps of `ibpm_amd.Batch`: stationary bodies (Cholesky, graph replay), moving bodies (plain CG,
  which the `ibpm` executable takes by default, and the preconditioned solve), the linearised and adjoint
  models.

Everything is FP64, the only precision whose forces hold the solver's 1e-6 accuracy; the library's FP32 and
BF16 transforms are measurement options and no program runs them.  Grids are those of ibpm_amd.workloads
and ragged ones; an FFT length takes factors 2, 3, 5 and at most 1024 cells per side, multiples of 4 with
more than one level.
"""
import functools
import math

import numpy as np
import torch

import ibpm_amd

RK3 = ((8 / 15, 0.0, 8 / 15), (5 / 12, -17 / 60, 2 / 3), (3 / 4, -5 / 12, 1.0))   # an, bn, cn of each substep


# ----------------------------------------------------------------- cases
def listed():
    return [
        # A single-level solve of a small grid: what one call costs.
        dict(name="poisson_64", kind="poisson", nx=64, ny=64, L=1),
        # One level, sides neither even nor alike.
        dict(name="helmholtz_225x150", kind="helmholtz", nx=225, ny=150, L=1),
        # The elliptic solve of a driver on the moving-plate grid.
        dict(name="poisson_512x5", kind="poisson", nx=512, ny=512, L=5),
        # The right-hand side of a substep on the cylinder grid (all stencils).
        dict(name="rhs_400x4", kind="rhs", nx=400, ny=400, L=4),
        # refreshState on a large ragged grid, transform lengths of no power of two.
        dict(name="flux_1000x600x5", kind="flux", nx=1000, ny=600, L=5),
        # The reference's standard run: a cylinder on one level, the wake in progress.
        dict(name="steps_cylinder_200", kind="steps", body="cylinder", flows=1, nx=200, ny=200, L=1, length=4.0,
             Re=100.0, dt=0.02, points=157, model="nonlinear", solver="cholesky", steps=10),
        # The same on four levels, 400 x 400.
        dict(name="steps_cylinder_400x4", kind="steps", body="cylinder", flows=1, nx=400, ny=400, L=4, length=4.0,
             Re=200.0, dt=0.01, points=314, model="nonlinear", solver="cholesky", steps=10),
        # A parameter sweep: uneven stationary flows advanced together.
        dict(name="steps_mixed_10x3", kind="steps", body="mixed", flows=10, nx=0, ny=0, L=3, length=4.0, Re=0.0,
             dt=0.005, points=0, model="nonlinear", solver="cholesky", steps=10),
        # One step of a linear stability code: the adjoint flow about a base state, on a ragged grid.
        dict(name="steps_adjoint_240x160x2", kind="steps", body="cylinder", flows=1, nx=240, ny=160, L=2, length=6.0,
             Re=60.0, dt=0.01, points=100, model="adjoint", solver="cholesky", steps=5),
        # A moving plate with the executable's default force solve (plain CG).
        dict(name="steps_plate_128x3", kind="steps", body="plate", flows=1, nx=128, ny=128, L=3, length=4.0, Re=300.0,
             dt=0.005, points=33, model="nonlinear", solver="cg", steps=2),
        # A moving plate, one flow, the preconditioned force solve.
        dict(name="steps_plate_512x5", kind="steps", body="plate", flows=1, nx=512, ny=512, L=5, length=4.0, Re=300.0,
             dt=0.0025, points=100, model="nonlinear", solver="tracked", steps=8),
        # Production: sixteen flows of three tandem plates advanced together.
        dict(name="steps_tandem_16x1024x6", kind="steps", body="tandem", flows=16, nx=1024, ny=1024, L=6, length=8.0,
             Re=500.0, dt=0.001, points=300, model="nonlinear", solver="tracked", steps=12),
    ]


def _sides(lo, hi, multiple):
    return [n for n in range(lo, hi + 1) if n % multiple == 0 and _smooth(n)]


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


def _near(rng, lo, hi, multiple):
    """A valid side in [lo, hi], spread over the logarithm."""
    s = _sides(lo, hi, multiple)
    want = math.exp(rng.uniform(math.log(s[0]), math.log(s[-1])))
    return min(s, key=lambda n: abs(n - want))


def draw(rng):
    kind = rng.choice(("poisson", "helmholtz", "flux", "rhs", "stationary", "stationary", "moving", "moving"))
    if kind in ("poisson", "helmholtz", "flux", "rhs"):
        L = rng.randint(1, 6)
        nx = _near(rng, 24, 1024, 1 if L == 1 else 4)
        ny = _near(rng, max(24, nx // 3), min(1024, 3 * nx), 1 if L == 1 else 4)
        return dict(kind=kind, nx=nx, ny=ny, L=L)
    if kind == "stationary":
        L = rng.randint(1, 4)
        nx = _near(rng, 96, 512, 4)
        ny = _near(rng, max(96, nx // 2), min(512, 2 * nx), 4)
        return dict(kind="steps", body="cylinder", flows=rng.choice((1, 1, 2, 4)), nx=nx, ny=ny, L=L,
                    length=4.0 * max(1.0, nx / ny), Re=rng.uniform(50, 200), dt=1.2 / max(nx, ny),
                    points=max(40, int(0.6 * math.pi * min(nx, ny) / 4)), model=rng.choice(("nonlinear", "linear")),
                    solver="cholesky", steps=rng.randint(3, 10))
    body = rng.choice(("plate", "tandem"))
    lo = 256 if body == "tandem" else 128
    n = _near(rng, lo, 1024, 4)
    solver = "cg" if n < 256 else "tracked"
    length = 8.0 if body == "tandem" else 4.0
    return dict(kind="steps", body=body, flows=1 if n < 256 else rng.randint(1, 6), nx=n, ny=n, L=rng.randint(2, 6),
                length=length, Re=rng.uniform(200, 500), dt=0.32 * length / n,
                points=(3 if body == "tandem" else 1) * int(0.78 * n / length), model="nonlinear", solver=solver,
                steps=2 if solver == "cg" else rng.randint(4, 8))


# --------------------------------------------------------------- geometry
def _points_body(xs, ys, more=""):
    return "body B\n" + "".join("  point %.17g %.17g\n" % p for p in zip(xs, ys)) + more + "end\n"


def _circle(n, r, x=0.0, y=0.0):
    a = 2 * math.pi * np.arange(n) / n
    return x + r * np.cos(a), y + r * np.sin(a)


def _ellipse(aspect, aoa, n):
    """n points, uniform in arc length, of an ellipse of major axis 1 rotated nose-up by aoa."""
    th = np.linspace(0, 2 * math.pi, 20001)
    seg = np.hypot(0.5 * np.diff(np.cos(th)), 0.5 / aspect * np.diff(np.sin(th)))
    s = np.concatenate([[0.0], np.cumsum(seg)])
    t = np.interp(np.arange(n) * s[-1] / n, s, th)
    x, y = 0.5 * np.cos(t), 0.5 / aspect * np.sin(t)
    c, si = math.cos(-aoa), math.sin(-aoa)
    return c * x - si * y, si * x + c * y


def _flows(case, seed):
    """The flows of a batch: (ibpm_amd.Flow, bodies), a body (xs, ys, x centre, pitch-plunge numbers or None)."""
    rng = np.random.default_rng([seed, 7])
    out = []
    for k in range(case["flows"]):
        nx, ny, Re, length = case["nx"], case["ny"], case["Re"], case["length"]
        bodies = []
        if case["body"] == "mixed":   # three sizes times three shapes
            nx = ny = (256, 384, 512)[k % 3]
            Re = float(rng.uniform(50, 300))
            dx, aoa = length / nx, math.radians(rng.uniform(0, 30))
            if k // 3 % 3 == 0:
                xy = _circle(int(math.pi * 0.5 / dx), 0.25, *rng.uniform(-0.1, 0.1, 2))
            elif k // 3 % 3 == 1:
                xy = _ellipse(float(rng.uniform(2, 5)), aoa, int(2.1 / dx))
            else:
                s = np.linspace(-0.5, 0.5, int(round(1 / dx)) + 1)
                xy = s * math.cos(aoa), -s * math.sin(aoa)
            bodies.append((xy[0], xy[1], 0.0, None))
        elif case["body"] == "cylinder":
            dx = length / nx
            r = case["points"] * dx / (2 * math.pi)   # points one cell apart
            x, y = rng.uniform(-0.1, 0.1, 2)
            bodies.append((*_circle(case["points"], r, x, y), 0.0, None))
        else:
            spacing = rng.uniform(1, 2)
            for xc in ((-spacing, 0.0, spacing) if case["body"] == "tandem" else (0.0,)):
                n = case["points"] // (3 if case["body"] == "tandem" else 1)
                mot = (math.radians(rng.uniform(5, 20)), rng.uniform(.2, .5), rng.uniform(.1, .3))
                y = rng.uniform(-0.05, 0.05)   # the plate's offset from its axis of rotation
                bodies.append((xc + np.linspace(-0.5, 0.5, n), np.full(n, y), xc, mot))
        geom = ""
        for xs, ys, xc, mot in bodies:
            more = "" if mot is None else ("  center %.17g 0\n  motion pitchplunge %.17g %.17g 0 %.17g %.17g 0\n"
                                           % (xc, mot[0], mot[1], mot[2], mot[1]))
            geom += _points_body(xs, ys, more)
        flow = ibpm_amd.Flow(nx, ny, case["L"], length, -length / 2, -length / 2 * ny / nx, Re, case["dt"], geom,
                             tol=1e-12 if case["solver"] == "cg" else 1e-10, model=case["model"])
        out.append((flow, bodies))
    return out


def _vortices(nx, ny, L, length, seed, device="cpu", count=24, spread=0.8):
    """A vorticity field of Gaussian vortices on every level (a wake in progress)."""
    rng = np.random.default_rng([seed, 11])
    half = spread * length / 2
    xc, yc, s, a = (torch.as_tensor(v, device=device)[:, None] for v in (
        rng.uniform(-half, half, count), rng.uniform(-half, half, count) * ny / nx,
        rng.uniform(0.04, 0.12, count) * length, 0.5 * rng.normal(size=count)))
    w = torch.empty(L, nx - 1, ny - 1, dtype=torch.float64, device=device)
    for lev in range(L):
        d = length / nx * 2 ** lev
        x = (torch.arange(1, nx, dtype=torch.float64, device=device) - nx / 2) * d
        y = (torch.arange(1, ny, dtype=torch.float64, device=device) - ny / 2) * d
        w[lev] = (a * torch.exp(-((x - xc) / s) ** 2)).T @ torch.exp(-((y - yc) / s) ** 2)   # separable
    return w


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


@functools.lru_cache(maxsize=1)
def _context():
    """One context for the program, as its owner keeps it."""
    return ibpm_amd.Context(0)


DX, DT, NU = 0.0125, 0.005, 0.01   # of the operator cases: finest spacing, step, viscosity
ALPHA = -0.5 * NU * DT             # Helmholtz: 1 + ALPHA Lap


def _base_state(case, seed):
    """Base state (vorticity, flux) of a linear model's flow, arrays of the flow's own grid."""
    w = _vortices(case["nx"], case["ny"], case["L"], case["length"], seed + 5, "cpu", 6)
    g = _Ref(case["nx"], case["ny"], case["L"], case["length"] / case["nx"])
    q = g.flux(g.solve(0, 0.0, -w), 1.0, 0.0)
    return w.numpy().ravel(), q.numpy().ravel()


def prepare(case, seed):
    nx, ny, L = case["nx"], case["ny"], case["L"]
    if case["kind"] != "steps":
        w = _vortices(nx, ny, L, DX * nx, seed, _device())
        s = dict(kind=case["kind"], ctx=_context(), args=(nx, ny, L, DX), w=w, out=torch.empty_like(w))
        nf = L * (2 * nx * ny + nx + ny)
        if case["kind"] == "flux":
            s["out"] = torch.empty(nf, dtype=torch.float64, device=w.device)
        if case["kind"] == "rhs":
            gen = torch.Generator(device=w.device).manual_seed(seed)
            s["q"] = DX * (1.0 + 0.1 * torch.randn(nf, dtype=torch.float64, device=w.device, generator=gen))
            s["nprev"] = _vortices(nx, ny, L, DX * nx, seed + 1, _device())
            s["n"] = torch.empty_like(w)
        return s
    flows = _flows(case, seed)
    b = ibpm_amd.Batch(_context(), [f for f, _ in flows])
    if case["model"] != "nonlinear":
        for k in range(len(flows)):
            b.set_base_state(*_base_state(case, seed + k), k=k)
    if case["solver"] == "tracked":
        b.set_precond("dense").set_precond_build("tracked", 0.1).set_warm_start("zero")
    b.init()
    if case["solver"] == "cholesky":
        b.use_graph()
    for k, (f, _) in enumerate(flows):
        b.set_omega(_vortices(f.nx, f.ny, f.ngrid, f.length, seed + 100 * k).numpy(), k)
    b.advance(2)   # the run is under way: its graph and its preconditioner are there
    return dict(kind="steps", batch=b, steps=case["steps"])


def run(s):
    if s["kind"] == "steps":
        b = s["batch"]
        b.advance(s["steps"])
        out = []
        for k in range(len(b.flows)):   # what a restart file holds
            out.append([b.omega(k), b.f(k)])
        if len(b.flows) == 1:
            out.append(b.q(0))
        return out
    lib, h = ibpm_amd.load(), s["ctx"].h
    nx, ny, L, dx = s["args"]
    w, out = s["w"].data_ptr(), s["out"].data_ptr()
    if s["kind"] == "poisson":
        rc = lib.ibpm_elliptic_solve(h, 0, nx, ny, L, dx, 0.0, w, out)
    elif s["kind"] == "helmholtz":
        rc = lib.ibpm_elliptic_solve(h, 1, nx, ny, L, dx, ALPHA, w, out)
    elif s["kind"] == "flux":
        rc = lib.ibpm_flux_from_vorticity(h, nx, ny, L, dx, 1.0, 0.1, w, out)
    else:
        rc = lib.ibpm_rhs(h, nx, ny, L, dx, DT, NU, 5 / 12, -17 / 60, s["q"].data_ptr(), w, s["nprev"].data_ptr(),
                          out, s["n"].data_ptr())
    if rc:
        raise ibpm_amd.IbpmError(lib.ibpm_last_error().decode())
    return [s["out"], s["n"]] if s["kind"] == "rhs" else s["out"]


def work(case):
    def solve_flops(g, nx, ny):   # two 2-D DSTs by FFT and the scaling
        return g * (2 * 2.5 * (math.log2(nx) + math.log2(ny)) + 6)

    if case["kind"] != "steps":
        nx, ny, L = case["nx"], case["ny"], case["L"]
        g, nf = L * (nx - 1) * (ny - 1), L * (2 * nx * ny + nx + ny)
        if case["kind"] == "rhs":
            return dict(bytes=8.0 * (4 * g + nf), flops=50.0 * g)
        return dict(bytes=8.0 * (2 * g if case["kind"] != "flux" else g + nf), flops=solve_flops(g, nx, ny))
    by = fl = 0.0
    for n in ([(384, 384)] * case["flows"] if case["body"] == "mixed" else [(case["nx"], case["ny"])] * case["flows"]):
        g = case["L"] * (n[0] - 1) * (n[1] - 1)
        # per substep: vorticity and the previous nonlinear term in and out, three solves over every level
        # and the stencils; the outputs once
        by += 8.0 * g * (4 * 3 * case["steps"] + 1)
        fl += 3 * case["steps"] * (3 * solve_flops(g, *n) + 50.0 * g)
    return dict(bytes=by, flops=fl)


# ------------------------------------------------------- the same in torch
class _Ref:
    """The operators on dense FP64 tensors: scalars [..., level, i, j], fluxes as (x, y) pairs of tensors
    [..., level, i, j]; sine transforms as matrix products."""

    def __init__(self, nx, ny, L, dx, device="cpu"):
        self.nx, self.ny, self.L, self.dx, self.dev = nx, ny, L, dx, device
        self.ex, self.ey = nx // 4, ny // 4

        def sines(n):
            k = torch.arange(1, n, dtype=torch.float64, device=device)
            return torch.sin(torch.outer(k, k).remainder(2 * n) * (math.pi / n)), 2 * (torch.cos(k * math.pi / n) - 1)
        self.sx, self.lx = sines(nx)
        self.sy, self.ly = sines(ny)

    def level_dx(self):
        return self.dx * 2.0 ** torch.arange(self.L, dtype=torch.float64, device=self.dev).view(-1, 1, 1)

    def inner(self):
        """Slices of the nodes strictly inside a coarse level's central region."""
        return slice(self.ex, self.ex + self.nx // 2 - 1), slice(self.ey, self.ey + self.ny // 2 - 1)

    def coarsify(self, f):
        f = f.clone()
        a, b = self.nx - 1, self.ny - 1
        for lev in range(1, self.L):
            s = lambda i, j: f[..., lev - 1, i:a - 2 + i:2, j:b - 2 + j:2]   # noqa: E731
            f[(..., lev, *self.inner())] = (0.25 * s(1, 1) + 0.125 * (s(2, 1) + s(1, 2) + s(0, 1) + s(1, 0))
                                            + 0.0625 * (s(2, 2) + s(2, 0) + s(0, 2) + s(0, 0)))
        return f

    def _ring(self, u, lev):
        """Boundary values of `lev` from the coarser solution u [..., level, i, j]: left, right, bottom, top."""
        if lev == self.L - 1:
            z = lambda n: torch.zeros(u.shape[:-3] + (n + 1,), dtype=u.dtype, device=u.device)   # noqa: E731
            return z(self.ny), z(self.ny), z(self.nx), z(self.nx)
        c = u[..., lev + 1, :, :]
        i0, i1, j0, j1 = self.ex - 1, self.ex - 1 + self.nx // 2, self.ey - 1, self.ey - 1 + self.ny // 2

        def refine(v):
            out = torch.empty(v.shape[:-1] + (2 * v.shape[-1] - 1,), dtype=v.dtype, device=v.device)
            out[..., ::2] = v
            out[..., 1::2] = 0.5 * (v[..., 1:] + v[..., :-1])
            return out
        return (refine(c[..., i0, j0:j1 + 1]), refine(c[..., i1, j0:j1 + 1]),
                refine(c[..., i0:i1 + 1, j0]), refine(c[..., i0:i1 + 1, j1]))

    def padded(self, u):
        """u with its boundary values: [..., level, 0..nx, 0..ny]."""
        p = torch.zeros(u.shape[:-2] + (self.nx + 1, self.ny + 1), dtype=u.dtype, device=u.device)
        p[..., 1:-1, 1:-1] = u
        for lev in range(self.L):
            p[..., lev, 0, :], p[..., lev, -1, :], p[..., lev, :, 0], p[..., lev, :, -1] = self._ring(u, lev)
        return p

    def solve(self, kind, alpha, f):
        """kind 0: Lap u = f; 1: (1 + alpha Lap) u = f; levels from coarse to fine."""
        f = self.coarsify(f)
        u = torch.zeros_like(f)
        for lev in reversed(range(self.L)):
            h2 = (self.dx * 2 ** lev) ** 2
            c = (1.0 if kind == 0 else alpha) / h2
            left, right, bottom, top = self._ring(u, lev)
            r = f[..., lev, :, :].clone()
            r[..., 0, :] -= c * left[..., 1:-1]
            r[..., -1, :] -= c * right[..., 1:-1]
            r[..., :, 0] -= c * bottom[..., 1:-1]
            r[..., :, -1] -= c * top[..., 1:-1]
            lam = (self.lx[:, None] + self.ly[None, :]) / h2
            hat = self.sx @ r @ self.sy / (lam if kind == 0 else 1 + alpha * lam)
            u[..., lev, :, :] = self.sx @ hat @ self.sy * (4.0 / (self.nx * self.ny))
        return u

    def curl(self, u):
        p = self.padded(u)
        return p[..., 1:] - p[..., :-1], p[..., :-1, :] - p[..., 1:, :]

    def join(self, x, y):
        return torch.cat([x.flatten(-2), y.flatten(-2)], -1)

    def split(self, q):   # q [..., level, flux]
        n = (self.nx + 1) * self.ny
        return (q[..., :n].unflatten(-1, (self.nx + 1, self.ny)), q[..., n:].unflatten(-1, (self.nx, self.ny + 1)))

    def flux(self, psi, u0, v0):
        x, y = self.curl(psi)
        d = self.level_dx()
        return self.join(x + u0 * d, y + v0 * d)

    def velocity(self, x, y):
        """Node velocities with the rules on the rim of each coarse level's central region."""
        d = self.level_dx()
        u = (x[..., 1:-1, 1:] + x[..., 1:-1, :-1]) / (2 * d)
        v = (y[..., 1:, 1:-1] + y[..., :-1, 1:-1]) / (2 * d)
        i0, i1, j0, j1 = self.ex, self.ex + self.nx // 2, self.ey, self.ey + self.ny // 2   # 1-based rim
        si, sj = self.inner()
        for lev in range(1, self.L):
            h = self.dx * 2 ** lev
            for j, jc, jf in ((j0, j0 - 1, 0), (j1, j1, self.ny - 1)):   # u on the rim's rows
                f = x[..., lev - 1, :, jf]
                u[..., lev, si, j - 1] = (x[..., lev, i0 + 1:i1, jc] * 2 / 3 + f[..., 2:-2:2] / 3
                                          + (f[..., 1:-3:2] + f[..., 3:-1:2]) / 6) / h
                other = x[..., lev, :, j if jc == j0 - 1 else j - 1]
                for i, fi in ((i0, 1), (i1, self.nx - 1)):
                    u[..., lev, i - 1, j - 1] = (x[..., lev, i, jc] * 8 + other[..., i] * 6 + f[..., fi] * 2) / 15 / h
            for i, ic, fi in ((i0, i0 - 1, 0), (i1, i1, self.nx - 1)):
                f = y[..., lev - 1, fi, :]
                v[..., lev, i - 1, sj] = (y[..., lev, ic, j0 + 1:j1] * 2 / 3 + f[..., 2:-2:2] / 3
                                          + (f[..., 1:-3:2] + f[..., 3:-1:2]) / 6) / h
                other = y[..., lev, i if ic == i0 - 1 else i - 1, :]
                for j, fj in ((j0, 1), (j1, self.ny - 1)):
                    v[..., lev, i - 1, j - 1] = (y[..., lev, ic, j] * 8 + other[..., j] * 6 + f[..., fj] * 2) / 15 / h
            u[..., lev, si, sj] = 0
            v[..., lev, si, sj] = 0
        return u, v

    def velocity_to_flux(self, a, b):
        """Fluxes of node values: x from a, y from b; the coarse levels' central fluxes from the finer level."""
        x = torch.zeros(a.shape[:-2] + (self.nx + 1, self.ny), dtype=a.dtype, device=a.device)
        y = torch.zeros(a.shape[:-2] + (self.nx, self.ny + 1), dtype=a.dtype, device=a.device)
        x[..., 1:-1, 1:-1] = 0.5 * (a[..., 1:] + a[..., :-1])
        y[..., 1:-1, 1:-1] = 0.5 * (b[..., 1:, :] + b[..., :-1, :])
        for lev in range(self.L):
            al, ar, ab, at = self._ring(a, lev)
            bl, br, bb, bt = self._ring(b, lev)
            x[..., lev, 1:-1, 0] = 0.5 * (a[..., lev, :, 0] + ab[..., 1:-1])
            x[..., lev, 1:-1, -1] = 0.5 * (a[..., lev, :, -1] + at[..., 1:-1])
            x[..., lev, 0, :] = 0.5 * (al[..., 1:] + al[..., :-1])
            x[..., lev, -1, :] = 0.5 * (ar[..., 1:] + ar[..., :-1])
            y[..., lev, 0, 1:-1] = 0.5 * (b[..., lev, 0, :] + bl[..., 1:-1])
            y[..., lev, -1, 1:-1] = 0.5 * (b[..., lev, -1, :] + br[..., 1:-1])
            y[..., lev, :, 0] = 0.5 * (bb[..., 1:] + bb[..., :-1])
            y[..., lev, :, -1] = 0.5 * (bt[..., 1:] + bt[..., :-1])
        x, y = x * self.level_dx(), y * self.level_dx()
        i0, i1, j0, j1 = self.ex, self.ex + self.nx // 2, self.ey, self.ey + self.ny // 2
        for lev in range(1, self.L):
            f, g = x[..., lev - 1, 2:-2:2, :], y[..., lev - 1, :, 2:-2:2]
            x[..., lev, i0 + 1:i1, j0:j1] = f[..., ::2] + f[..., 1::2]
            y[..., lev, i0:i1, j0 + 1:j1] = g[..., ::2, :] + g[..., 1::2, :]
        return x, y

    def curl_of_flux(self, x, y):
        return (y[..., 1:, 1:-1] - y[..., :-1, 1:-1] + x[..., 1:-1, :-1] - x[..., 1:-1, 1:]) / self.level_dx() ** 2

    def cross(self, q, w):
        u, v = self.velocity(*self.split(q))
        return self.velocity_to_flux(v * w, -u * w)

    def laplacian(self, w):
        return -self.curl_of_flux(*self.curl(w))

    def nonlinear(self, model, q, w, base):
        if model == "nonlinear":
            return self.curl_of_flux(*self.cross(q, w))
        w0, q0 = base
        if model == "linear":
            return self.curl_of_flux(*self.cross(q0, w)) + self.curl_of_flux(*self.cross(q, w0))
        (u0, v0), (u, v) = self.velocity(*self.split(q0)), self.velocity(*self.split(q))
        return self.laplacian(self.coarsify(u0 * v - u * v0)) - self.curl_of_flux(*self.cross(q, w0))


def _delta(r):
    near = (1 + torch.sqrt((1 - 3 * r * r).clamp(min=0))) / 3
    far = (5 - 3 * r - torch.sqrt((1 - 3 * (1 - r) ** 2).clamp(min=0))) / 6
    return torch.where(r <= 0.5, near, torch.where(r < 1.5, far, torch.zeros_like(r)))


class _Body:
    """Interpolation between the level-0 fluxes and points (E and its transpose)."""

    def __init__(self, g, x, y, xoff, yoff):
        self.g, h = g, g.dx
        idx, wgt = [], []
        o = torch.arange(-2, 4, device=g.dev)
        for d in (0, 1):
            fx, fy = (x - xoff) / h, (y - yoff) / h
            i, j = torch.floor(fx)[:, None].long() + o, torch.floor(fy)[:, None].long() + o
            wi = _delta((i + 0.5 * d - fx[:, None]).abs())
            wj = _delta((j + 0.5 * (1 - d) - fy[:, None]).abs())
            at = i[:, :, None] * (g.ny + d) + j[:, None, :] + d * (g.nx + 1) * g.ny
            idx.append(at.flatten(1))
            wgt.append((wi[:, :, None] * wj[:, None, :]).flatten(1))
        self.idx, self.wgt = torch.cat(idx), torch.cat(wgt)

    def gather(self, q):   # q [..., level, flux]
        return (q[..., 0, :][..., self.idx] * self.wgt).sum(-1) / self.g.dx

    def smear(self, f):    # Curl E^T f
        g = self.g
        q = torch.zeros(f.shape[:-1] + (2 * g.nx * g.ny + g.nx + g.ny,), dtype=f.dtype, device=f.device)
        q.index_add_(-1, self.idx.flatten(), (f[..., :, None] * self.wgt).flatten(-2) * g.dx)
        x, y = g.split(q)
        out = torch.zeros(f.shape[:-1] + (g.L, g.nx - 1, g.ny - 1), dtype=f.dtype, device=f.device)
        out[..., 0, :, :] = (y[..., 1:, 1:-1] - y[..., :-1, 1:-1] + x[..., 1:-1, :-1] - x[..., 1:-1, 1:]) / g.dx ** 2
        return out


def _exact_flow(case, flow, bodies, w, base_state, nsteps):
    """The state after nsteps of one flow: [vorticity, force], flux."""
    g = _Ref(flow.nx, flow.ny, flow.ngrid, flow.length / flow.nx, _device())
    t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=g.dev)   # noqa: E731
    linear = case["model"] != "nonlinear"
    base = None
    if linear:
        w0, q0 = base_state
        base = (t(w0).view(g.L, g.nx - 1, g.ny - 1), t(q0).view(g.L, -1))
    w = w.to(g.dev)
    u0 = 0.0 if linear else 1.0
    q = g.flux(g.solve(0, 0.0, -w), u0, 0.0)
    n_prev, time, fixed = None, 0.0, {}
    for _ in range(nsteps):
        for i, (an, bn, cn) in enumerate(RK3):
            now, beta, nu = time + cn * flow.dt, (an + bn) * flow.dt, 1.0 / flow.Re
            alpha = -0.5 * beta * nu
            moving = any(m is not None for *_, m in bodies)
            if moving or i not in fixed:
                px, py, pu, pv = [], [], [], []
                for xs, ys, xc, m in bodies:
                    th = thd = hy = hv = 0.0
                    if m is not None:
                        om = 8.0 * math.atan(1.0) * m[1]
                        th, thd = m[0] * math.sin(om * now), m[0] * om * math.cos(om * now)
                        hy, hv = m[2] * math.sin(om * now), m[2] * om * math.cos(om * now)
                    a, c, s = xs - xc, math.cos(th), math.sin(th)
                    px.append(a * c - ys * s + xc)
                    py.append(hy + a * s + ys * c)
                    pu.append(-a * s * thd - ys * c * thd)
                    pv.append(a * c * thd - ys * s * thd + hv)
                E = _Body(g, t(np.concatenate(px)), t(np.concatenate(py)), flow.xoffset, flow.yoffset)
                n = E.idx.shape[0]
                cols = []
                eye = torch.eye(n, dtype=torch.float64, device=g.dev)
                for k in range(0, n, 64):
                    psi = g.solve(0, 0.0, -g.solve(1, alpha, beta * E.smear(eye[k:k + 64])))
                    cols.append(E.gather(g.join(*g.curl(psi))))
                still = t(np.concatenate(pu + pv))
                uniform = torch.zeros(g.L, 2 * g.nx * g.ny + g.nx + g.ny, dtype=torch.float64, device=g.dev)
                uniform[0, :(g.nx + 1) * g.ny] = u0 * g.dx
                M = torch.cat(cols).T
                if case["solver"] == "cholesky":   # factored from its upper triangle
                    M = M.triu() + M.triu(1).T
                fixed[i] = E, torch.linalg.lu_factor(M), still - E.gather(uniform)
            E, M, b = fixed[i]
            N = g.nonlinear(case["model"], q, w, base)
            a = w + flow.dt * (0.5 * nu * (an + bn) * g.laplacian(w) + an * N + bn * (N if n_prev is None else n_prev))
            n_prev = N
            ws = g.solve(1, alpha, a)
            rhs = E.gather(g.join(*g.curl(g.solve(0, 0.0, -ws)))) - b
            f = torch.linalg.lu_solve(*M, rhs[:, None])[:, 0]
            w = ws - g.solve(1, alpha, beta * E.smear(f))
            q = g.flux(g.solve(0, 0.0, -w), u0, 0.0)
        time += flow.dt
    return [w.flatten(), f], q.flatten()


def exact(case, seed):
    nx, ny, L = case["nx"], case["ny"], case["L"]
    if case["kind"] != "steps":
        g = _Ref(nx, ny, L, DX, _device())
        s = prepare(case, seed)
        w = s["w"]
        if case["kind"] == "poisson":
            return g.solve(0, 0.0, w)
        if case["kind"] == "helmholtz":
            return g.solve(1, ALPHA, w)
        if case["kind"] == "flux":
            return g.flux(g.solve(0, 0.0, -w), 1.0, 0.1).flatten()
        an, bn = 5 / 12, -17 / 60
        N = g.nonlinear("nonlinear", s["q"].view(L, -1), w, None)
        return [w + DT * (0.5 * NU * (an + bn) * g.laplacian(w) + an * N + bn * s["nprev"]), N]
    # the force matrix takes two solves per unknown, once, or per substep where the body moves
    builds = 3 * (case["steps"] + 2 if case["solver"] != "cholesky" else 1)
    n = max(nx, ny, 400 if case["body"] == "mixed" else 0)
    unknowns = 2 * (case["points"] or 250)
    if case["flows"] * builds * unknowns * 2 * L * 8.0 * n ** 3 > 1.5e14:
        return None
    out = []
    for k, (flow, bodies) in enumerate(_flows(case, seed)):
        w = _vortices(flow.nx, flow.ny, flow.ngrid, flow.length, seed + 100 * k)
        base = _base_state(case, seed + k) if case["model"] != "nonlinear" else None
        state, q = _exact_flow(case, flow, bodies, w, base, case["steps"] + 2)
        out.append(state)
        if case["flows"] == 1:
            out.append(q)
    return out
