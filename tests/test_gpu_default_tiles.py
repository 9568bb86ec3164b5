"""Tiles that a solver starts out with (chosen by grid size) against the
128-byte, 8-row tiles on 32-lane Z lines: the same discrete solution, so the
states after three steps agree to rounding (FP64 1e-12, FP32 1e-5, relative to
the velocity norm; the bars of the parity tests with a margin).  Sizes either
side of each line of the rule, and a batch of mixed grids."""
import numpy as np
import pytest

from cmcx import domains
from cmcx.solver import make_batch, make_solver
from gpu_util import rel_l2_scaled, say, vel_norm

pytestmark = pytest.mark.gpu

SHAPES = [(32, 32, 32), (64, 21, 33), (65, 32, 32), (40, 40, 40), (86, 75, 82), (12, 9, 95), (12, 9, 96),
          (12, 9, 128), (12, 9, 129), (256, 40, 64), (90, 25, 40), (189, 60, 20), (130, 129, 8)]


def _same(a, b, dtype):
    vs = vel_norm(*a[:3])
    tol = 1e-12 if dtype == "f64" else 1e-5
    for x, y, sc in zip(a, b, (vs, vs, vs, 0.0, 0.0)):
        assert np.isfinite(x).all()
        assert rel_l2_scaled(x, y, sc) < tol


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_default_tiles(shape, dtype):
    d = domains.random_domain(shape, np.random.default_rng(1), 0.1, free_faces=True)
    d.dt = 1e-3
    say(f"[default tiles] {shape} {dtype}")
    got = []
    for plain in (False, True):
        s = make_solver(d, dtype, path=1)
        if plain:
            for a in range(3):
                s.set_tile_variant(a, 0)
        s.run(3, d.dt, 2, 1)
        got.append(s.fields())
        s.close()
    _same(*got, dtype)


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_default_tiles_batch(dtype):
    rng = np.random.default_rng(2)
    ds = [domains.random_domain(s, rng, 0.1) for s in ((20, 30, 24), (7, 5, 100), (96, 90, 100), (33, 12, 9))]
    got = []
    for plain in (False, True):
        s = make_batch(ds, dtype)
        if plain:
            for a in range(3):
                s.set_tile_variant(a, 0)
        s.run(2, 1e-3, 2, 1)
        got.append([s.fields_of(i) for i in range(len(ds))])
        s.close()
    for a, b in zip(*got):
        _same(a, b, dtype)
