"""2D line solves in chunks where an error in c', d' or x hardly shrinks from row to
row, so that the lanes' early starts leave many chunks to be run again: stiff
viscous rows (c' to 0.999), and flows of up to 200 cells per step, which the
estimate behind the early starts does not see.  Whole steps against the oracle: the
iterations, the error in FP64, and the state bit for bit in FP64, to 1e-5 in FP32.
Every step is accepted, but for those of the last test."""
import ctypes

import numpy as np
import pytest

import oracle_lib
from cmcx import _lib, domains
from cmcx.params import FluidParams
from cmcx.solver import AdiSolver2D
from gpu_util import rel_l2, say

pytestmark = pytest.mark.gpu


def _flow(nx, ny, u, dt):
    """A channel whose fluid starts at the inlet's profile, with waves in v and T."""
    d = domains.channel2d(nx, ny, radius=ny / 10, centre=(nx * 0.3, ny * 0.5), u_max=u, dt=dt)
    t, vx, vy, T = (a.reshape(nx, ny) for a in (d.type, d.vx, d.vy, d.T))
    i, j = np.arange(nx)[:, None] / nx, np.arange(ny)[None, :] / ny
    inn = t == domains.NODE_IN
    vx[inn] = np.broadcast_to(vx[0].copy(), t.shape)[inn]
    vy[inn] = (0.02 * np.sin(5 * i) * np.sin(6.28 * j))[inn]
    T[inn] = (T + 0.01 * np.cos(9 * i) * np.sin(4 * j))[inn]
    return d


def _step(s, dt, G, L):
    err, it = ctypes.c_double(0.0), ctypes.c_int(0)
    rc = _lib.lib().cmcx2d_step(s.h, dt, G, L, ctypes.byref(err), ctypes.byref(it))
    return rc, err.value, it.value


def _run(d, dtype, G, L, steps, accepted):
    p = FluidParams.normalized(d.re, 0.72, 1.4)
    s = AdiSolver2D(dtype).Init(d, p)
    o = oracle_lib.Oracle2D(d, dtype, p)
    for k in range(steps):
        s.UpdateBoundaries()
        o.update_boundaries()
        r, rerr, rit = o.step(d.dt, G, L)
        rc, err, it = _step(s, d.dt, G, L)
        say(f"  step {k}: {rc} err {err:.3e} ({rerr:.3e}) iterations {it}")
        assert (r == 0) == (rc == 0) == accepted
        assert it == rit
        if dtype == "f64":  # (in FP32 the oracle's own sum of some 10^4 terms is 10^4 2^-24 off)
            np.testing.assert_allclose(err, rerr, rtol=1e-9)
        if not accepted:
            break
    u, v, _, T = s.fields()
    for nm, a, b in zip("uvT", (u, v, T), o.layer(0)):
        if dtype == "f64":
            assert np.array_equal(a, b), nm
        else:
            assert rel_l2(a, b) < 1e-5, nm
    s.close()


# (nx, ny, dt, steps): c' of constant rows 0.94 to 0.998
STIFF = [(256, 40, 1.0, 2), (130, 70, 0.3, 2), (40, 50, 0.3, 2), (33, 36, 0.3, 2), (500, 36, 1.0, 2)]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("L", [1, 2])
@pytest.mark.parametrize("nx,ny,dt,steps", STIFF)
def test_stiff_rows(nx, ny, dt, steps, L, dtype):
    _run(_flow(nx, ny, 0.02, dt), dtype, 2, L, steps, True)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,dt", [(256, 40, 10.0), (130, 70, 100.0), (500, 36, 100.0)])
def test_stiffest_rows(nx, ny, dt, dtype):
    _run(_flow(nx, ny, 0.02, dt), dtype, 2, 1, 1, True)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,cells", [(200, 50, 5), (200, 50, 10), (300, 40, 20), (400, 33, 20)])
def test_fast_flows(nx, ny, cells, dtype):
    _run(_flow(nx, ny, cells / (nx - 1) / 1e-3, 1e-3), dtype, 2, 1, 1, True)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,cells,dt", [(200, 50, 15, 1e-3), (300, 40, 200, 1e-3), (33, 36, 6.4, 10.0)])
def test_refused_steps(nx, ny, cells, dt, dtype):
    """Errors above 1 in a later iteration, in the first, and of stiff rows."""
    _run(_flow(nx, ny, cells / (nx - 1) / dt, dt), dtype, 2, 1, 1, False)
