"""Workloads of the fluid solvers, as a user's program runs them: inputs, one
pass, the work a pass cannot do without, and the pass's results in 64 bits.

A case is a dict of plain values; "kind" says which solver it drives:

  step     one 3D grid (AdiSolver3D): a run of time steps from a given state,
           then the fields u, v, w, p, T on the device
  output   the reference's driver loop: every `every` steps the layer is read
           back resampled (GetLayer), the fields at the end
  batch    several independent 3D grids advanced together (BatchSolver3D)
  adjoint  a recorded rollout and its gradients (adjoint_forward / _backward)
  adi2d    the 2D ADI solver: a whole run from its initial state
  stable2d the 2D projection solver: a whole run from its initial state

A 3D pass starts from the state given in `prepare` (the program writes it
through the state's device pointers, as a rollout, a parameter study or a
restart does), so every pass does the same work.  The 2D solvers have no entry
point that replaces their state: there a pass is the whole run, creation
included.
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cmc-fluid-solver_amd"))

from cmcx import domains  # noqa: E402
from cmcx.params import FluidParams  # noqa: E402
from cmcx.solver import AdiSolver2D, StableSolver2D, make_batch, make_solver  # noqa: E402

IN, OUT, BOUND, VALVE = 0, 1, 2, 3
FREE = 1


def listed():
    return [
        # a small box as the smallest grids of a parameter study: launches count
        dict(name="lid32_f32", kind="step", flow="lid", nx=32, ny=32, nz=32, dtype="f32", steps=20,
             G=4, L=1, dt=1e-3, re=300.0, graph=False, tune=False),
        # a small box stepped as a replayed graph, the option for launch-bound loops
        dict(name="lid64_f32_graph", kind="step", flow="lid", nx=64, ny=64, nz=64, dtype="f32", steps=10,
             G=4, L=1, dt=1e-3, re=300.0, graph=True, tune=False),
        # a grid as geometry files give them: odd sides, FP64, two local iterations
        dict(name="channel75_odd_f64", kind="step", flow="channel", nx=75, ny=51, nz=67, dtype="f64",
             steps=10, G=4, L=2, dt=5e-4, re=400.0, graph=False, tune=False),
        # the 128^3 lid-driven box with a sphere, in both field types
        dict(name="lid128_f32", kind="step", flow="lid", nx=128, ny=128, nz=128, dtype="f32", steps=10,
             G=4, L=1, dt=5e-4, re=400.0, graph=False, tune=False),
        dict(name="lid128_f64", kind="step", flow="lid", nx=128, ny=128, nz=128, dtype="f64", steps=5,
             G=4, L=1, dt=5e-4, re=400.0, graph=False, tune=False),
        # the headline workload: 256^3 channel with ellipsoids, tiles autotuned as the benchmark does
        dict(name="ellipsoids256_f32", kind="step", flow="channel", nx=256, ny=256, nz=256, dtype="f32",
             steps=5, G=4, L=1, dt=2e-4, re=1000.0, graph=False, tune=True),
        # a large channel of ragged sides, default tiles
        dict(name="channel_ragged_f32", kind="step", flow="channel", nx=250, ny=203, nz=187, dtype="f32",
             steps=4, G=4, L=1, dt=2e-4, re=1000.0, graph=False, tune=False),
        # the driver loop with results read back for the output file every fifth step
        dict(name="output_loop_f32", kind="output", flow="channel", nx=128, ny=96, nz=112, dtype="f32",
             steps=10, every=5, out=50, G=4, L=2, dt=5e-4, re=400.0, graph=False, tune=False),
        # 64 independent boxes in one launch per sweep
        dict(name="batch64_f32", kind="batch", count=64, edges="32,48,64,96", pick=0, dtype="f32", steps=10,
             G=4, L=1, dt=1e-3, graph=False, tune=True),
        # gradient of a probe's kinetic energy with respect to inlet, state and parameters
        dict(name="adjoint96_f32", kind="adjoint", n=96, dtype="f32", steps=40, every=8, G=4, dt=3e-3),
        # the 2D channel with a cylinder, FP64
        dict(name="channel2d_f64", kind="adi2d", nx=256, ny=128, dtype="f64", steps=20, G=4, L=1, dt=1e-3),
        # the 2D projection solver on a box with an inflow and an outflow in one wall
        dict(name="pipe2d_f64", kind="stable2d", nx=120, ny=135, dtype="f64", steps=1, G=2),
    ]


def _side(rng, lo, hi):
    """A side between lo and hi, spread over the logarithm; odd ones as likely as even ones."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("step", "output", "batch", "adjoint", "adi2d", "stable2d"),
                       weights=(10, 2, 2, 3, 2, 1))[0]
    dtype = rng.choice(("f32", "f32", "f64"))
    w = 1 if dtype == "f32" else 2
    if kind in ("step", "output"):
        c = dict(kind=kind, flow=rng.choice(("lid", "channel")), nx=_side(rng, 24, 256), ny=_side(rng, 24, 256),
                 nz=_side(rng, 24, 256), dtype=dtype, G=rng.choice((2, 4)), L=rng.choice((1, 1, 2)),
                 dt=rng.choice((2e-4, 5e-4)), re=float(rng.choice((200, 400, 1000))),
                 graph=rng.random() < 0.3, tune=rng.random() < 0.2)
        cells = c["nx"] * c["ny"] * c["nz"] * w * c["L"]
        c["steps"] = max(2, min(20, int(4 * 256 ** 3 / cells)))
        if kind == "output":
            c["steps"] = max(2, c["steps"] // 2)
            c["every"] = rng.choice((1, 2, 5))
            c["out"] = rng.choice((0, 32, 50)) if cells < 4e6 else rng.choice((32, 50))
        return c
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(4, 48), edges=rng.choice(("32,48,64,96", "33,45,63,80", "24,40,72")),
                    pick=rng.randint(1, 1000), dtype=dtype, steps=rng.randint(3, 10) // w, G=4, L=1, dt=rng.choice((5e-4, 1e-3)),
                    graph=rng.random() < 0.5, tune=rng.random() < 0.5)
    if kind == "adjoint":
        return dict(kind="adjoint", n=3 * rng.randint(8, 32), dtype=dtype, steps=rng.randint(8, 30 // w),
                    every=rng.randint(2, 10), G=rng.choice((2, 4)), dt=rng.choice((1e-3, 2e-3, 3e-3)))
    if kind == "adi2d":
        return dict(kind="adi2d", nx=_side(rng, 64, 320), ny=_side(rng, 48, 200), dtype=dtype,
                    steps=rng.randint(5, 20), G=rng.choice((2, 4)), L=rng.choice((1, 1, 2)), dt=1e-3)
    return dict(kind="stable2d", nx=rng.randint(40, 110), ny=rng.randint(40, 120), dtype=dtype, steps=1, G=2)


# -- inputs ---------------------------------------------------------------------------


def _np(dtype):
    return np.float32 if dtype == "f32" else np.float64


def _torch(dtype):
    return torch.float32 if dtype == "f32" else torch.float64


def _box(case, rng):
    """A lid-driven box or a channel (inlet u = 1 at x = 0, free outlet) with a few ellipsoids removed."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["flow"] == "channel" and nx == ny == nz == 256:
        d = domains.ellipsoids(nx, seed=int(rng.integers(1 << 30)))
    else:
        d = domains.box(nx, ny, nz)
        m = min(nx, ny, nz)
        solid = np.zeros((nx, ny, nz), bool)
        for _ in range(1 if case["flow"] == "lid" else 6):
            ax = rng.uniform(0.10, 0.25, 3) * m
            c = [rng.uniform(0.2, 0.8) * (n - 1) for n in (nx, ny, nz)]
            x, y, z = [((np.arange(n) - c[k]) / ax[k]) ** 2 for k, n in enumerate((nx, ny, nz))]
            solid |= x[:, None, None] + y[None, :, None] + z[None, None, :] < 1.0
        inner = solid.ravel()
        d.type[inner] = BOUND
        if case["flow"] == "lid":
            d.vx.reshape(nx, ny, nz)[:, :, -1] = 1.0
        else:
            t, bv, bt = (a.reshape(nx, ny, nz) for a in (d.type, d.bc_vel, d.bc_temp))
            t[0] = t[-1] = VALVE
            bv[-1] = bt[-1] = FREE
            d.vx.reshape(nx, ny, nz)[0] = 1.0
    d.re, d.dt = case["re"], case["dt"]
    return d


def _shapes(case):
    """Sides of a batch's grids: part of the case, not of its inputs."""
    r = random.Random(case["pick"])
    e = [int(x) for x in case["edges"].split(",")]
    return [tuple(r.choice(e) for _ in range(3)) for _ in range(case["count"])]


def _batch(case, rng):
    """Lid-driven boxes with one to three spheres each, every one with its own Reynolds number."""
    ds = []
    for s in _shapes(case):
        d = domains.box(*s)
        solid = np.zeros(s, bool)
        for _ in range(int(rng.integers(1, 4))):
            r = rng.uniform(0.10, 0.30) * min(s)
            x, y, z = [(np.arange(n) - rng.uniform(1, n - 2)) ** 2 for n in s]
            solid |= x[:, None, None] + y[None, :, None] + z[None, None, :] < r * r
        d.type[solid.ravel()] = BOUND
        d.vx.reshape(s)[:, :, -1] = 1.0
        d.re, d.dt = float(rng.uniform(50, 500)), case["dt"]
        ds.append(d)
    return ds


def _flow(d, rng, u0):
    """A smooth flow on the fluid nodes of a grid: u0 along x and a few waves; the node values elsewhere."""
    s = d.shape
    fields = []
    for k, base in enumerate((u0, 0.0, 0.0, d.base_t)):
        f = np.full(s, base, np.float32)
        for _ in range(2):
            a = rng.uniform(0.02, 0.05) * (1.0 if k < 3 else 0.2)
            w = [np.sin(rng.uniform(1, 4) * math.pi * np.linspace(0, 1, n) + rng.uniform(0, 6.28)).astype(np.float32)
                 for n in s]
            f += (a * w[0])[:, None, None] * (w[1][:, None] * w[2][None, :])[None]
        fields.append(f.ravel())
    inside = d.type == IN
    return [np.where(inside, f, g.astype(np.float32)) for f, g in zip(fields, (d.vx, d.vy, d.vz, d.T))]


def _grids(case, seed):
    """The grids of a 3D case and the state each starts from (numpy, 32-bit values)."""
    rng = np.random.default_rng([seed, 17])
    if case["kind"] == "batch":
        ds = _batch(case, rng)
    elif case["kind"] == "adjoint":
        n = case["n"]
        ds = [domains.cylinder_channel(n, radius=n / 8, seed=int(rng.integers(1 << 30)), dt=case["dt"])[0]]
    else:
        ds = [_box(case, rng)]
    lid = case["kind"] == "batch" or case.get("flow") == "lid"
    return ds, [_flow(d, rng, 0.0 if lid else 0.8) for d in ds]


class _Pointer:
    """A device address as torch takes it (no copy)."""

    def __init__(self, address, n, dtype):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4" if dtype == "f32" else "<f8",
                                         "data": (address, False), "version": 2}


def _channel2d(case, seed):
    rng = np.random.default_rng([seed, 23])
    nx, ny = case["nx"], case["ny"]
    return domains.channel2d(nx, ny, radius=ny / 8, centre=(nx * rng.uniform(0.2, 0.4), ny * rng.uniform(0.4, 0.6)),
                             u_max=rng.uniform(0.8, 1.1), dt=case["dt"])


def _pipe2d(case, seed):
    """A walled box of 0.7 mm cells, outside cells around it, with an inflow in one half of its right wall and
    the outflow in the other."""
    rng = np.random.default_rng([seed, 29])
    nx, ny = case["nx"], case["ny"]
    t = np.full((nx, ny), OUT, np.uint8)
    t[2:-2, 2:-2] = BOUND
    t[3:-3, 3:-3] = IN
    vx = np.zeros((nx, ny))
    m, v = int(ny * rng.uniform(0.38, 0.44)), 0.1 * rng.uniform(0.9, 1.1)  # the same flow in and out
    vx[-3, 3:3 + m] = v
    vx[-3, -3 - m:-3] = -v
    return domains.Domain2D(nx, ny, 0.0007, 0.0007, 1.0, t.ravel(), np.zeros(nx * ny, np.uint8), vx.ravel(),
                            np.zeros(nx * ny), np.ones(nx * ny), dt=0.035 / 30)


def prepare(case, seed):
    if case["kind"] == "adi2d":
        return dict(case=case, grid=_channel2d(case, seed))
    if case["kind"] == "stable2d":
        return dict(case=case, grid=_pipe2d(case, seed))
    ds, init = _grids(case, seed)
    ty, n = _torch(case["dtype"]), sum(d.n for d in ds)
    if case["kind"] == "batch":
        s = make_batch(ds, case["dtype"])
    else:
        s = make_solver(ds[0], case["dtype"], path=1)
    if case.get("tune"):
        s.autotune()
    if case.get("graph"):
        s.set_graph(True)
    start = [torch.from_numpy(np.concatenate([q[f] for q in init])).to("cuda").to(ty) for f in range(4)]
    st = dict(case=case, solver=s, sizes=[d.n for d in ds], start=start,
              out=torch.zeros(5, n, dtype=ty, device="cuda"))
    if case["kind"] == "adjoint":
        ids = torch.from_numpy(_probe(case["n"])).to("cuda")
        st.update(probe=ids, seed=torch.zeros(4, n, dtype=ty, device="cuda"),
                  gbar=torch.zeros(4, n, dtype=ty, device="cuda"), sbar=torch.zeros(4, n, dtype=ty, device="cuda"))
    return st


def _probe(n):
    """Nodes of a cube behind the cylinder, centred in y and z."""
    m = max(2, n // 6)
    x = np.arange(n // 2 + 1, n // 2 + 1 + m)
    y = np.arange(n // 2 - m // 2, n // 2 - m // 2 + m)
    return ((x[:, None, None] * n + y[None, :, None]) * n + y[None, None, :]).ravel()


# -- one pass -------------------------------------------------------------------------


def _rows(t):
    return [t[f].data_ptr() for f in range(t.shape[0])]


def _each_grid(state):
    """(index, slice of the flat arrays) of every grid, selected in turn in a batch."""
    s, o = state["solver"], 0
    for i, n in enumerate(state["sizes"]):
        if len(state["sizes"]) > 1:
            s.select(i)
        yield i, slice(o, o + n)
        o += n


def _restart(state):
    """The state `prepare` made, written through the solver's device pointers."""
    for _, at in _each_grid(state):
        for p, v in zip(state["solver"].state_ptrs(), state["start"]):
            q = v[at]
            torch.as_tensor(_Pointer(p, q.numel(), state["case"]["dtype"]), device="cuda").copy_(q)


def _read(state):
    """u, v, w, p, T of every grid into the program's own device arrays."""
    out = state["out"]
    for _, at in _each_grid(state):
        state["solver"].fields_device(*_rows(out[:, at]))
    return dict(zip("uvwpT", out))


def run(state):
    c = state["case"]
    if c["kind"] in ("adi2d", "stable2d"):
        d = state["grid"]
        if c["kind"] == "adi2d":
            s, dt = AdiSolver2D(c["dtype"]), c["dt"]
            s.Init(d, FluidParams.normalized(d.re, domains.PR, domains.LAMBDA))
        else:
            s, dt = StableSolver2D(c["dtype"]), d.dt
            s.Init(d, FluidParams.dimensional(0.05, 1000.0, 287.0, 0.0257, 1000.0))
        iters = 0
        for _ in range(c["steps"]):
            s.UpdateBoundaries()
            iters += s.TimeStep(dt, c["G"], c.get("L", 1))[1]
        u, v, p, T = s.fields()
        s.close()
        return dict(u=u, v=v, p=p, T=T, iters=iters)
    s = state["solver"]
    _restart(state)
    if c["kind"] == "adjoint":
        s.adjoint_forward(c["steps"], c["dt"], c["G"], c["every"])
        final = _read(state)
        ids, seed = state["probe"], state["seed"]
        for f, name in enumerate("uvw"):
            seed[f, ids] = final[name][ids] / ids.numel()
        pbar = s.adjoint_backward_device(_rows(seed), _rows(state["gbar"]), _rows(state["sbar"]))
        return dict(final=final, gbar=state["gbar"], sbar=state["sbar"], pbar=pbar.astype(_np(c["dtype"])))
    if c["kind"] == "output":
        layers = []
        for i in range(c["steps"]):
            s.UpdateBoundaries()
            s.TimeStep(c["dt"], c["G"], c["L"], i % 10 == 0)
            if (i + 1) % c["every"] == 0:
                vel, T = s.GetLayer(c["out"], c["out"], c["out"])
                layers.append((vel, T.astype(_np(c["dtype"]))))  # T holds values of the field type
        return dict(layers=layers, final=_read(state))
    s.run(c["steps"], c["dt"], c["G"], c["L"])
    return dict(final=_read(state))


# -- what a pass cannot do without ----------------------------------------------------

# per node and sweep: the interior row of four fields (about 60), the elimination of
# two matrices with four right-hand sides and the back substitution (about 30)
SWEEP_FLOPS = 90


def work(case):
    w = 4 if case["dtype"] == "f32" else 8
    k = case["kind"]
    if k in ("adi2d", "stable2d"):
        n = case["nx"] * case["ny"]
        per = 2 * 70 * case.get("L", 1) if k == "adi2d" else 60  # a projection's relaxation depends on the flow
        return dict(bytes=n * (3 * 8 + 2 + 4 * w), flops=float(n) * case["steps"] * case["G"] * per)
    if k == "batch":
        n = sum(a * b * c for a, b, c in _shapes(case))
    else:
        n = case["n"] ** 3 if k == "adjoint" else case["nx"] * case["ny"] * case["nz"]
    sweeps = 3.0 * case["G"] * case.get("L", 1) * case["steps"]
    if k == "adjoint":  # reversed sweeps: the transposed solve and the transposed stencils
        return dict(bytes=n * ((4 + 5 + 4 + 4 + 4) * w + 1), flops=n * sweeps * (SWEEP_FLOPS + 160))
    return dict(bytes=n * ((4 + 5) * w + 1), flops=n * sweeps * SWEEP_FLOPS)


# -- the same in 64 bits --------------------------------------------------------------


def _shift(x, k, axis):
    """x at the neighbour k rows on along an axis (the edge rows wrap; their values are not used)."""
    return torch.roll(x, -k, axis)


def _pcr(a, b, c, d, axis):
    """Tridiagonal systems along an axis by parallel cyclic reduction; d carries the right-hand sides first."""
    n = a.shape[axis]
    s = 1
    at = torch.arange(n, device=a.device).reshape([-1 if k == axis else 1 for k in range(a.dim())])
    a, c, d = a / b, c / b, d / b
    while s < n:
        lo, hi = at >= s, at < n - s
        al, cr = torch.where(lo, a, 0), torch.where(hi, c, 0)
        am, cm = _shift(a, -s, axis), _shift(c, -s, axis)
        ap, cp = _shift(a, s, axis), _shift(c, s, axis)
        r = 1.0 / (1.0 - al * cm - cr * ap)
        d = (d - al * _shift(d, -s, axis + 1) - cr * _shift(d, s, axis + 1)) * r
        a, c = -al * am * r, -cr * cp * r
        s *= 2
    return d


class _Lines(torch.autograd.Function):
    """x with tridiag(a, b, c) x = d along an axis, and its gradients by the transposed systems."""

    @staticmethod
    def forward(ctx, a, b, c, d, axis):
        x = _pcr(a, b, c, d, axis)
        ctx.save_for_backward(a, b, c, x)
        ctx.axis = axis
        return x

    @staticmethod
    def backward(ctx, g):
        a, b, c, x = ctx.saved_tensors
        ax = ctx.axis
        lam = _pcr(_shift(c, -1, ax), b, _shift(a, 1, ax), g, ax)
        return (-(lam * _shift(x, -1, ax + 1)).sum(0), -(lam * x).sum(0), -(lam * _shift(x, 1, ax + 1)).sum(0), lam, None)


class _Model3D:
    """The 3D time step as dense tensor arithmetic: every grid line one tridiagonal system."""

    def __init__(self, d, device):
        s = d.shape
        t = torch.from_numpy(d.type.reshape(s)).to(device)
        self.inside, self.fixed = t == IN, (t == BOUND) | (t == VALVE)
        self.h = (d.dx, d.dy, d.dz)
        self.free = [torch.from_numpy(a.reshape(s).astype(bool)).to(device) for a in (d.bc_vel, d.bc_temp)]
        self.values = torch.stack([torch.from_numpy(a.reshape(s)) for a in (d.vx, d.vy, d.vz, d.T)]).to(device)
        self.first, self.last, self.both = [], [], []
        for ax in range(3):
            n = s[ax]
            at = torch.arange(n, device=device).reshape([-1 if k == ax else 1 for k in range(3)])
            nxt = _shift(self.inside, 1, ax) & (at < n - 1) & ~self.inside
            prv = _shift(self.inside, -1, ax) & (at > 0) & ~self.inside
            self.both.append(nxt & prv)
            self.first.append(nxt & ~prv)
            self.last.append(prv & ~nxt)

    def _d(self, x, ax):
        return (_shift(x, 1, ax) - _shift(x, -1, ax)) / (2 * self.h[ax])

    def sweep(self, ax, src, temp, g, prm, dt):
        """The solution on the nodes of the axis's systems (other nodes: zero), the four fields."""
        vT, nu, kappa, phi_c = prm
        inside, h = self.inside, self.h[ax]
        adv = temp[ax] / (2 * h)
        own = [self._d(temp[f], ax) for f in range(3)]
        phi = sum((2 if f == ax else 1) * own[f] * own[f] for f in range(3))
        for o in range(3):
            if o != ax:
                phi = phi + own[o] * self._d(temp[ax], o)
        out = []
        for q, (vis, fields) in enumerate(((nu / h ** 2, (0, 1, 2)), (kappa / h ** 2, (3,)))):
            fa, fb = self.first[ax] & self.free[q], self.last[ax] & self.free[q]
            value = (self.first[ax] | self.last[ax] | self.both[ax]) & ~fa & ~fb
            fa_, fb_, both_ = (x.double() for x in (fa, fb, fa | fb))
            a = torch.where(inside, -adv - vis, -fb_)
            c = torch.where(inside, adv - vis, -fa_)
            b = torch.where(inside, (3 / dt + 2 * vis) * torch.ones_like(both_), 1.0 + both_)
            d = []
            for f in fields:
                r = 3 / dt * src[f]
                if f == ax:
                    r = r - vT * self._d(temp[3], ax)
                if f == 3:
                    r = r + phi_c * phi
                d.append(torch.where(inside, r, torch.where(value, g[f], 0.0)))
            out.append(_Lines.apply(a, b, c, torch.stack(d), ax))
        return torch.cat(out)

    def step(self, state, g, prm, dt, G, L):
        cur = torch.where(self.fixed, g, state)
        nxt, temp = cur, cur
        for _ in range(G):
            src = cur
            for ax in (2, 1, 0):
                x = None
                for _ in range(L):
                    x = self.sweep(ax, src, temp, g, prm, dt)
                    temp = torch.where(self.inside, (temp + x) / 2, temp)
                ends = self.inside | self.first[ax] | self.last[ax] | self.both[ax]
                if ax != 1:
                    nxt = torch.where(ends, x, nxt)
                src = x
            temp = torch.where(self.inside, (temp + x) / 2, temp)
        return nxt


def _channel2d_run(case, seed):
    """The 2D run line by line over whole arrays (Thomas along each direction)."""
    d = _channel2d(case, seed)
    nx, ny, L, dt = case["nx"], case["ny"], case["L"], case["dt"]
    p = FluidParams.normalized(d.re, domains.PR, domains.LAMBDA)
    t, bc = d.type.reshape(nx, ny), d.bc.reshape(nx, ny)
    g = np.stack([d.vx.reshape(nx, ny), d.vy.reshape(nx, ny), d.T.reshape(nx, ny)])
    h = (d.dx, d.dy)
    inner = np.zeros((nx, ny), bool)
    inner[:-1, :-1] = True
    inm = inner & (t == IN)
    spans = []
    for ax in (0, 1):  # first and last node of every line's system
        m = t if ax == 0 else t.T
        n = m.shape[0]
        a, b = np.full(m.shape[1], n), np.full(m.shape[1], -1)
        for j in range(m.shape[1]):
            f = np.flatnonzero((m[:-1, j] != OUT) & (m[1:, j] == IN))
            r = np.flatnonzero((m[1:, j] != OUT) & (m[:-1, j] == IN))
            if len(f) and len(r):
                a[j], b[j] = f[0], r[-1] + 1
        spans.append((a, b))

    def diff(x, ax):
        r = np.zeros_like(x)
        lo, hi = [slice(None)] * 2, [slice(None)] * 2
        mid = list(lo)
        lo[ax], hi[ax], mid[ax] = slice(None, -2), slice(2, None), slice(1, -1)
        r[tuple(mid)] = (x[tuple(hi)] - x[tuple(lo)]) / (2 * h[ax])
        return r

    def direction(ax, lc, temp, out):
        tl = np.where(inner, temp, 0.0)
        first, last = spans[ax]
        n = (nx, ny)[ax]
        at = np.arange(n)[:, None]
        row = (at > first) & (at < last)
        ends = [(at == first), (at == last)]
        turn = (lambda x: x) if ax == 0 else (lambda x: x.T)
        nl = np.zeros_like(tl)
        for it in range(L):
            u, v, T = tl
            src = [np.zeros((nx, ny)) for _ in range(3)]
            src[ax] = -p.v_T * diff(T, ax)
            du = [diff(u, ax), diff(v, ax)]
            src[2] = p.t_phi * (2 * du[ax] ** 2 + du[1 - ax] ** 2 + du[1 - ax] * diff(tl[ax], 1 - ax))
            w = turn(tl[ax]) / (2 * h[ax])
            fr = turn(bc) == FREE
            for f in range(3):
                vis = (p.t_vis if f == 2 else p.v_vis) / h[ax] ** 2
                a = np.where(row, -w - vis, np.where(ends[1] & fr, 1.0, 0.0))
                c = np.where(row, w - vis, np.where(ends[0] & fr, -1.0, 0.0))
                b = np.where(row, 1 / dt + 2 * vis, np.where(ends[1] & fr, -1.0, 1.0))
                r = np.where(row, turn(lc[f] / dt + src[f]), np.where((ends[0] | ends[1]) & ~fr, turn(g[f]), 0.0))
                cp, dp = np.zeros_like(a), np.zeros_like(a)
                cp[0], dp[0] = c[0] / b[0], r[0] / b[0]
                for i in range(1, n):
                    den = b[i] - a[i] * cp[i - 1]
                    cp[i], dp[i] = c[i] / den, (r[i] - a[i] * dp[i - 1]) / den
                for i in range(n - 2, -1, -1):
                    dp[i] -= cp[i] * dp[i + 1]
                nl[f] = turn(np.where(row | ends[0] | ends[1], dp, turn(nl[f])))
            tl = np.where(inm, nl if it == 0 else (tl + nl) / 2, tl)
        return np.where(inm, tl, temp), np.where(inm, nl, out)

    cells = (t[:-1, :-1] == IN) & (t[1:, :-1] == IN) & (t[:-1, 1:] == IN) & (t[1:, 1:] == IN)
    cur, iters = g.copy(), 0
    for _ in range(case["steps"]):
        cur = np.where((t == BOUND) | (t == VALVE), g, cur)
        nxt, half, temp = (np.where(inner, cur, 0.0) for _ in range(3))
        err, it = 1.0, 0
        while it < case["G"] or err > 0.1:
            temp, half = direction(0, cur, temp, half)
            temp, nxt = direction(1, half, temp, nxt)
            u, v = nxt[0], nxt[1]
            tx = h[1] * (u[1:, :-1] - u[:-1, :-1]) + (u[1:, 1:] - u[:-1, 1:]) / 2
            ty = h[0] * (v[:-1, 1:] - v[:-1, :-1]) + (v[1:, 1:] - v[1:, :-1]) / 2
            err = float(np.abs(tx + ty)[cells].mean())
            temp = np.where(inm, nxt if it == 0 else (temp + nxt) / 2, temp)
            it += 1
            if it > 100 or not err <= 1.0:
                raise RuntimeError("the run leaves the range that the solver accepts")
        cur = np.where(inner, nxt, cur)
        iters += it
    return dict(u=cur[0].ravel(), v=cur[1].ravel(), p=p.v_T * cur[2].ravel(), T=cur[2].ravel(), iters=None)


def _final(x, prm):
    u = x.reshape(4, -1)
    return dict(u=u[0], v=u[1], w=u[2], p=prm[0] * u[3], T=u[3])


def exact(case, seed):
    k = case["kind"]
    if k == "adi2d":
        return _channel2d_run(case, seed)
    if k == "stable2d":
        return None  # thousands of cell-ordered relaxation sweeps: minutes in numpy
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    ds, init = _grids(case, seed)
    finals = []
    for d, q in zip(ds, init):
        m, fp = _Model3D(d, dev), d.params()
        g = m.values
        x = torch.stack([torch.from_numpy(a).to(dev).double().reshape(d.shape) for a in q])
        prm = torch.tensor([fp.v_T, fp.v_vis, fp.t_vis, fp.t_phi], dtype=torch.float64, device=dev)
        if k == "adjoint":
            return _exact_gradient(case, m, g, x, prm)
        layers = []
        for i in range(case["steps"]):
            old = torch.where(m.fixed, g, x)
            x = m.step(x, g, prm, case["dt"], case["G"], case["L"])
            if k == "output" and (i + 1) % case["every"] == 0:
                # the layer that is read back is the state before the step
                at = [torch.arange(case["out"] or n, device=dev) * n // (case["out"] or n) for n in d.shape]
                o = old[:, at[0]][:, :, at[1]][:, :, :, at[2]].reshape(4, -1)
                layers.append((o[:3].T.contiguous(), o[3]))
        finals.append(_final(x, prm))
        if k == "output":
            return dict(layers=layers, final=finals[0])
    return dict(final={f: torch.cat([x[f] for x in finals]) for f in "uvwpT"})


def _exact_gradient(case, m, g, x, prm):
    from torch.utils.checkpoint import checkpoint

    g, x0, prm = (v.clone().requires_grad_(True) for v in (g, x, prm))
    x = x0
    for _ in range(case["steps"]):
        x = checkpoint(m.step, x, g, prm, case["dt"], case["G"], 1, use_reentrant=False)
    ids = torch.from_numpy(_probe(case["n"])).to(x.device)
    inside = m.inside.reshape(-1)[ids]
    u = x.reshape(4, -1)[:3, ids] * inside
    (0.5 * (u ** 2).sum() / ids.numel()).backward()
    n = case["n"] ** 3
    return dict(final=_final(x.detach(), prm.detach()), gbar=g.grad.reshape(4, n), sbar=x0.grad.reshape(4, n),
                pbar=prm.grad)
