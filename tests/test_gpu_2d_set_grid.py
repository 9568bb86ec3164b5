"""New cell types between the steps of the 2D solvers (SetGrid): the lists that
follow them, against the oracle."""
import numpy as np
import pytest

import oracle_lib
from cmcx.params import FluidParams
from cmcx.solver import StableSolver2D
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
