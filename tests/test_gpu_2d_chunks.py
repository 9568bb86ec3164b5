"""The 2D line solve in chunks (k2_sweep_chunks) against the oracle: FP64 bit
for bit, FP32 to 1e-5 (the bars of the 2D tests), at line lengths either side
of a chunk, of 4- and 8-row chunks and of the longest line that it takes, with
rows that shrink an error fast, slowly (chunks run again many times) and hardly
at all (solved serially), one and two inner iterations, and states that blow
up."""
import numpy as np
import pytest

import oracle_lib
from cmcx import _lib, domains
from cmcx.params import FluidParams
from cmcx.solver import AdiSolver2D
from gpu_util import rel_l2, say

pytestmark = pytest.mark.gpu


def _check(d, p, dtype, steps, G, L, what):
    s = AdiSolver2D(dtype).Init(d, p)
    o = oracle_lib.Oracle2D(d, dtype, params=p)
    for _ in range(steps):
        s.UpdateBoundaries()
        o.update_boundaries()
        r, _, ito = o.step(d.dt, G, L)
        try:
            _, it = s.TimeStep(d.dt, G, L)
        except _lib.CmcxError:
            it = None
        assert (it is None) == (r != 0)
        if it is None:
            break
        assert it == ito
    u, v, _, T = s.fields()
    for nm, a, b in zip("uvT", (u, v, T), o.layer(0)):
        say(f"  {what}: {nm} {rel_l2(a, b):.2e}")
        if dtype == "f64":
            assert np.array_equal(a, b, equal_nan=True), nm
        else:
            assert rel_l2(a, b) < 1e-5, nm
    s.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(48, 40), (61, 64), (64, 65), (129, 33), (200, 255), (256, 57), (257, 64),
                                   (320, 200), (512, 20), (513, 34)])
def test_line_lengths(shape, dtype):
    nx, ny = shape
    d = domains.channel2d(nx, ny, radius=ny / 8, centre=(nx * 0.3, ny * 0.5), dt=1e-3)
    _check(d, FluidParams.normalized(d.re, 0.72, 1.4), dtype, 2, 3, 1, f"{shape} {dtype}")


@pytest.mark.parametrize("L", [1, 2])
@pytest.mark.parametrize("dt", [1e-5, 1e-3, 4e-3, 1e-2, 1e-1])
def test_time_steps(dt, L):
    d = domains.channel2d(130, 70, radius=9.0, centre=(40, 35), dt=dt, u_max=0.1)
    _check(d, FluidParams.normalized(d.re, 0.72, 1.4), "f64", 2, 2, L, f"dt {dt} L {L}")


@pytest.mark.parametrize("u_max", [30.0, 3e3, 1e200])
def test_fast_flows(u_max):
    """Advection far above the viscous estimate that sets the early starts, up
    to infinities."""
    d = domains.channel2d(200, 50, radius=6.0, centre=(60, 25), dt=1e-3, u_max=u_max)
    _check(d, FluidParams.normalized(d.re, 0.72, 1.4), "f64", 1, 1, 1, f"u_max {u_max}")


@pytest.mark.parametrize("vis", [0.0, 1e-12])
def test_no_viscosity(vis):
    d = domains.channel2d(90, 50, radius=6.0, centre=(30, 25), dt=1e-3)
    _check(d, FluidParams(1.0, vis, vis, 0.0), "f64", 2, 2, 1, f"vis {vis}")
