"""Relaxations of one to a few sweeps on grids whose rows are shorter than a turn of
the fronts, whose steps end with the last column: against the oracle, bit for bit, states
and sweep counts."""
import pytest

from test_gpu_relaxation_fronts import _run
from test_stable2d_pins import walled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("tol", [1e3, 0.9, 0.3, 0.05])
@pytest.mark.parametrize("shape", [(6, 6), (7, 5), (12, 10), (20, 58), (20, 59), (65, 27), (65, 63), (130, 9), (300, 12)])
def test_few_sweeps(shape, tol, dtype):
    _run(walled(*shape, 4, out_corner=min(shape) > 12, obstacles=2), dtype, tol, f"{shape} {dtype} {tol}", G=2)
