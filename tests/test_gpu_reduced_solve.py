"""The reduced systems of the fused sweeps end their reduction when the rows of a
work-group (Z: of a wavefront) no longer depend on one another.  Lines of 128 to
256 nodes whose off-diagonal to diagonal ratio lets that happen after 0, 1, 2, 3
or none of the steps (per-row decay 0.003, 0.03, 0.31, 0.57 and 0.87), every
tile variant, against the oracle with the bars of the other parity tests (1e-11
in FP64, 1e-5 in FP32: the worst matrix here, of condition 216, loses less)."""
import numpy as np
import pytest

from cmcx import domains
from gpu_util import say
from test_gpu_batch import _check_batch
from test_gpu_edges import FUSED, _compare, _long

pytestmark = pytest.mark.gpu

# (Re, dt): nu / h^2 is about 100 on lines of 128 nodes at Re 160
CASES = [(160.0, 1e-4), (160.0, 1e-3), (160.0, 2e-2), (160.0, 1e-1), (10.0, 1e-1)]


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("re,dt", CASES)
@pytest.mark.parametrize("shape", [(128, 7, 20), (7, 128, 20), (6, 7, 200)])
def test_coupling(shape, re, dt, dtype):
    d = _long(shape, 11)
    d.dx = d.dy = d.dz = 1.0 / 127.0
    d.re, d.dt = re, dt
    say(f"[coupling] {shape} {dtype} Re={re} dt={dt}")
    variants = [(v, v, min(v, 7)) for v in range(10)] if shape[2] < 100 else [(0, 0, v) for v in range(8)]
    _compare(d, dtype, FUSED, variants, steps=1)


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_mixed_batch(dtype):
    """Coupled and decoupled grids in one launch, several tiles to a work-group."""
    rng = np.random.default_rng(8)
    doms = [domains.random_domain(s, rng, 0.1) for s in ((96, 20, 40), (33, 90, 35), (17, 12, 70))]
    for d, re in zip(doms, (10.0, 1e4, 160.0)):
        d.re, d.dt = re, 2e-2
    say(f"[coupling batch] {dtype}")
    _check_batch(doms, dtype, FUSED, steps=1)
