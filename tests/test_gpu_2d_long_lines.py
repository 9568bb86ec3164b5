"""2D steps whose lines are too long for the solve in chunks in one direction, the
other or both (over 512 rows), where the Picard layer's second copy is kept by a
copy instead of the X solve, and grids of more cells than the 65536 threads of the
divergence sums: against the oracle, FP64 bit for bit, FP32 to 1e-5
(the bars of the 2D tests), several Picard iterations and steps."""
import pytest

from cmcx import domains
from cmcx.params import FluidParams
from test_gpu_2d_chunks import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(512, 40), (514, 40), (40, 514), (530, 517)])
def test_directions(shape, dtype):
    nx, ny = shape
    d = domains.channel2d(nx, ny, radius=min(nx, ny) / 8, centre=(nx * 0.3, ny * 0.5), dt=1e-3)
    _check(d, FluidParams.normalized(d.re, 0.72, 1.4), dtype, 2, 4, 1, f"{shape} {dtype}")


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(257, 256), (331, 199), (300, 409)])
def test_many_cells(shape, dtype):
    nx, ny = shape
    d = domains.channel2d(nx, ny, radius=min(nx, ny) / 8, centre=(nx * 0.3, ny * 0.5), dt=1e-3)
    _check(d, FluidParams.normalized(d.re, 0.72, 1.4), dtype, 2, 3, 1, f"{shape} {dtype}")
