"""The Stable solver's relaxation with q in LDS by anti-diagonals (k2s_poisson_lds)
against the oracle, bit for bit, states and sweep counts, at the sizes where
its layout changes: one and several wavefronts of rows, rows shorter than the
members' lag, the largest grid that fits, the first that does not (the other
kernel), masks with many boundary cells on one diagonal, relaxations of
fewer sweeps than a group and of several launches, and sweep caps."""
import numpy as np
import pytest

import oracle_lib
from cmcx import _lib
from cmcx._lib import CmcxError
from cmcx.params import FluidParams
from cmcx.solver import StableSolver2D
from gpu_util import say
from test_gpu_stable2d import _same_state
from test_stable2d_pins import BOUND, IN, OUT, domain, walled

pytestmark = pytest.mark.gpu

P = FluidParams(1.0, 0.02, 0.0, 0.0)


def _run(t, dtype, tol, what, steps=1, G=1):
    d = domain(t, 0.01, 0.012, seed=3)
    o = oracle_lib.Oracle2D(d, dtype, P, method="stable")
    s = StableSolver2D(dtype).Init(d, P)
    o.set_poisson(tol, 1 << 30)
    s.set_poisson(tol)
    for k in range(steps):
        s.UpdateBoundaries()
        o.update_boundaries()
        try:
            _, it = s.TimeStep(2e-4, G, 1)
        except CmcxError:  # the divergence error may pass 1.0: in both
            it = None
        r, _, rit = o.step(2e-4, G, 1)
        assert (it is None) == (r != 0)
        sw = list(s.poisson_sweeps())
        say(f"  {what}: sweeps {sw}")
        assert sw == list(o.poisson_sweeps())
        _same_state(s, o, what)
        if it is None:
            break
    s.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(6, 6), (63, 20), (64, 58), (64, 59), (65, 27), (128, 60), (129, 40), (193, 24),
                                   (300, 12), (512, 7), (30, 300), (9, 1500), (118, 166), (118, 168), (150, 40)])
def test_sizes(shape, dtype):
    """118 x 166 FP64 fills the LDS, 118 x 168 does not; rows beyond the turn length
    (65 x 27 and on) have wavefronts with delays of their own."""
    _run(walled(*shape, 4, out_corner=min(shape) > 12, obstacles=min(shape) // 2), dtype, 0.03, f"{shape} {dtype}")


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_many_boundary_cells(dtype):
    """Every second cell a wall (all the boundary cells of a diagonal in one
    step), and a region without fluid."""
    t = walled(70, 50, 1, out_corner=False, obstacles=0)
    ii, jj = np.indices(t.shape)
    t[(t == IN) & ((ii + jj) % 2 == 0)] = BOUND
    t[:10] = OUT
    t[10] = BOUND
    _run(t, dtype, 0.02, f"chequered {dtype}", steps=2)


@pytest.mark.parametrize("tol", [0.5, 0.05, 1e-4, 1e-7])
def test_sweep_counts(tol):
    """From a few sweeps to more than one launch of 2048."""
    _run(walled(40, 44, 2, obstacles=6), "f64", tol, f"tol {tol}")


@pytest.mark.parametrize("cap", [1, 7, 16, 17, 2048, 2049])
def test_sweep_cap(cap):
    """A relaxation that meets its cap leaves the sweeps it did and the error."""
    d = domain(walled(60, 58, 2, obstacles=6), 0.01, 0.012, seed=3)
    s = StableSolver2D("f64").Init(d, P)
    s.set_poisson(1e-300, cap)
    s.UpdateBoundaries()
    with pytest.raises(CmcxError) as e:
        s.TimeStep(2e-4, 1, 1)
    assert e.value.code == _lib.CMCX_ERR_PICARD
    assert list(s.poisson_sweeps()) == [cap]
    s.close()
