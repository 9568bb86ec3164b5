"""The adjoint's tape is laid out once: a second recording on the same solver
(after new node values, another number of Picard iterations or steps, a release,
a replaced state) gives the gradients of a fresh solver, exactly."""
import numpy as np
import pytest

from cmcx import domains
from cmcx.solver import make_solver
from gpu_util import say

pytestmark = pytest.mark.gpu

DT = 1e-3


def _domain(seed):
    d = domains.random_domain((12, 10, 14), np.random.default_rng(4), 0.1, free_faces=True)
    r = np.random.default_rng(seed)
    wall = d.type != domains.NODE_IN
    for a in (d.vx, d.vy, d.vz):
        a[wall] = 0.1 * r.normal(size=int(wall.sum()))
    d.T[wall] = 1.0 + 0.01 * r.normal(size=int(wall.sum()))
    d.re, d.dt = 50.0, DT
    return d


def _gradient(s, start, steps, G, every):
    s.set_fields(*start)
    s.adjoint_forward(steps, DT, G, every)
    seed = np.random.default_rng(9).normal(size=(4, s.grid.n)) * (s.grid.type == domains.NODE_IN)
    return s.adjoint_backward(seed)


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("second", [dict(), dict(G=3), dict(G=1), dict(steps=5), dict(steps=2), dict(every=1)])
@pytest.mark.parametrize("change", ["values", "release", "none"])
def test_second_recording(dtype, second, change):
    a, b = _domain(1), _domain(2)
    if change != "values":
        b = a
    run = dict(steps=4, G=2, every=2)
    s = make_solver(a, dtype, path=1)
    _gradient(s, (a.vx, a.vy, a.vz, a.T), **run)
    if change == "release":
        s.adjoint_release()
    if change == "values":
        s.set_boundary(b.bc_vel, b.bc_temp, b.vx, b.vy, b.vz, b.T)
    run.update(second)
    got = _gradient(s, (b.vx, b.vy, b.vz, b.T), **run)
    fresh = make_solver(b, dtype, path=1)
    want = _gradient(fresh, (b.vx, b.vy, b.vz, b.T), **run)
    say(f"[adjoint tape] {dtype} {change} {run}")
    for g, w in zip(got, want):
        assert np.isfinite(w).all() and np.abs(w).max() > 0
        assert np.array_equal(g, w)
    s.close()
    fresh.close()
