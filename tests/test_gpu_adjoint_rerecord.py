"""A rollout recorded again over a tape that an earlier recording used, where the
sweeps left other values on nodes that are not NODE_IN: grids with NODE_OUT nodes
whose state holds GetLayer's 99999 there, and free ends, recorded on one path and
then on the other.  The gradients are those of a solver that records for the first
time, bit for bit."""
import numpy as np
import pytest

from cmcx import domains
from cmcx.solver import make_solver
from gpu_util import say

pytestmark = pytest.mark.gpu


def _grid():
    d = domains.random_domain((14, 11, 19), np.random.default_rng(9), 0.1, free_faces=True)
    t = d.type.reshape(d.shape)
    t[:3] = domains.NODE_OUT
    t[3] = domains.NODE_BOUND
    t[9:, 8:, :] = domains.NODE_OUT
    t[8, 7:, :] = t[8:, 7, :] = domains.NODE_BOUND
    return d


def _record(s, start, seed):
    s.set_fields(*start)
    s.adjoint_forward(5, 1e-3, 2, 2)
    return (*s.adjoint_backward(seed), *s.fields())


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("paths", [(1, 1), (1, 0), (0, 1)])
def test_over_an_older_tape(paths, dtype):
    d = _grid()
    a = make_solver(d, dtype, path=paths[0])
    a.run(2, 1e-3, 2, 1)
    start = [a.fields()[k] for k in (0, 1, 2, 4)]
    seed = np.random.default_rng(1).standard_normal((4, d.n))
    say(f"[recorded again] {paths} {dtype}")
    _record(a, start, seed)
    for _ in range(3):  # the fill into either state buffer, and recorded with it
        a.GetLayer()
        a.run(1, 1e-3, 2, 1)
    a.adjoint_forward(5, 1e-3, 2, 2)
    a.adjoint_backward(seed)
    if paths[1] != paths[0]:
        a.set_options(path=paths[1])
    b = make_solver(d, dtype, path=paths[1])
    for x, y in zip(_record(a, start, seed), _record(b, start, seed)):
        assert np.array_equal(x, y)
    a.close()
    b.close()
