"""New cell types between the steps of the 2D solvers (SetGrid): the lists that
follow them, and types that are refused, against the oracle."""
import numpy as np
import pytest

import oracle_lib
from cmcx import _lib, domains
from cmcx.params import FluidParams
from cmcx.solver import AdiSolver2D, StableSolver2D
from gpu_util import say
from test_gpu_stable2d import _steps
from test_stable2d_pins import BOUND, IN, domain, walled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(60, 50), (130, 170)])
def test_stable_boundary_lists_grow_and_shrink(shape, dtype):
    """Few, many (every second cell) and few boundary cells again, with q in LDS (60 x
    50) and per span (130 x 170 FP64)."""
    few = walled(*shape, 3, out_corner=False, obstacles=2)
    many = few.copy()
    ii, jj = np.indices(shape)
    many[(many == IN) & ((ii + jj) % 2 == 0) & (ii > shape[0] // 2)] = BOUND
    other = walled(*shape, 5, obstacles=9)
    masks = [few, many, other, many, few]
    p = FluidParams(1.0, 0.02, 0.0, 0.0)
    ds = [domain(t, 0.01, 0.012, seed=3) for t in masks]
    o = oracle_lib.Oracle2D(ds[0], dtype, p, method="stable")
    s = StableSolver2D(dtype).Init(ds[0], p)
    o.set_poisson(0.1, 1 << 30)
    s.set_poisson(0.1)
    grids = lambda k: (ds[k].type, ds[k].bc, ds[k].vx, ds[k].vy, ds[k].T)  # noqa: E731
    _steps(s, o, 2e-5, 1, len(masks), f"{shape} {dtype}", grids)
    s.close()


@pytest.mark.parametrize("ny", [24, 600])
@pytest.mark.parametrize("L", [1, 2])
def test_adi_goes_on_after_refused_types(ny, L):
    """A column whose only NODE_IN cell lies on the grid's edge has no line system
    of two nodes: refused, and the steps that follow are those of the types
    before it; then types that are taken."""
    nx = 30
    p = FluidParams.normalized(100.0, 0.72, 1.4)
    ds = [domains.channel2d(nx, ny, radius=r, centre=(12, 11), dt=1e-3) for r in (4.0, 6.0, 2.0)]
    bad = np.full((nx, ny), BOUND, np.uint8)
    bad[2:-2, 2:-2] = IN
    bad[-1, 1] = IN
    o = oracle_lib.Oracle2D(ds[0], "f64", params=p)
    s = AdiSolver2D("f64").Init(ds[0], p)
    for k, d in enumerate((None, None, ds[1], None, ds[2])):
        if d is not None:
            o.set_grid(d.type, d.bc, d.vx, d.vy, d.T)
            s.SetGrid(d.type, d.bc, d.vx, d.vy, d.T)
        else:
            with pytest.raises(_lib.CmcxError) as e:
                s.SetGrid(bad, ds[0].bc, ds[0].vx, ds[0].vy, ds[0].T)
            assert e.value.code == _lib.CMCX_ERR_ARG
        s.UpdateBoundaries()
        o.update_boundaries()
        r, _, it = o.step(1e-3, 2, L)
        assert r == 0
        assert s.TimeStep(1e-3, 2, L)[1] == it
        u, v, _, T = s.fields()
        for nm, a, b in zip("uvT", (u, v, T), o.layer(0)):
            assert np.array_equal(a, b), (k, nm)
        say(f"  step {k}: equal")
    s.close()
