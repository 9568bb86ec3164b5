"""Calls that the device refuses: what comes after them."""
import numpy as np
import pytest

from cmcx import _lib, domains
from cmcx.solver import make_solver
from gpu_util import say

pytestmark = pytest.mark.gpu

# checkpoints or a tape of terabytes: the allocation fails at once
TOO_MUCH = [dict(steps=2_000_000_000, checkpoint_every=1), dict(steps=2_000_000_000, checkpoint_every=100_000_000)]


def _solver(dtype="f32"):
    d = domains.random_domain((9, 8, 12), np.random.default_rng(6), 0.1)
    s = make_solver(d, dtype, path=1)
    s.run(2, 1e-3, 2, 1)
    return s


@pytest.mark.parametrize("how", TOO_MUCH)
def test_the_next_solver(how):
    """A failed call's error is reported by that call and by no later one."""
    a = _solver()
    say(f"[failed calls] {how}")
    with pytest.raises(_lib.CmcxError) as e:
        a.adjoint_forward(dt=1e-3, num_global=2, **how)
    assert e.value.code == _lib.CMCX_ERR_HIP
    b = _solver()
    for x, y in zip(a.fields(), b.fields()):
        assert np.array_equal(x, y)
    a.close()
    b.close()


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("how", TOO_MUCH)
def test_adjoint_after_a_failed_recording(how, dtype):
    """A recording too large for the device leaves none, and a smaller one after it
    (than the one before it, too) gives the gradients of a solver that never tried."""
    a, b = _solver(dtype), _solver(dtype)
    seed = np.random.default_rng(1).standard_normal((4, a.grid.n))
    a.adjoint_forward(6, 1e-3, 2, 2)
    a.adjoint_backward(seed)
    b.run(6, 1e-3, 2, 1)
    say(f"[failed recording] {how} {dtype}")
    with pytest.raises(_lib.CmcxError) as e:
        a.adjoint_forward(dt=1e-3, num_global=2, **how)
    assert e.value.code == _lib.CMCX_ERR_HIP
    assert a.adjoint_generation() == 0
    with pytest.raises(_lib.CmcxError) as e:
        a.adjoint_backward(seed)
    assert e.value.code == _lib.CMCX_ERR_STATE
    a.set_fields(*(b.fields()[k] for k in (0, 1, 2, 4)))
    b.set_fields(*(b.fields()[k] for k in (0, 1, 2, 4)))
    for s in (a, b):
        s.adjoint_forward(4, 1e-3, 2, 2)
    for x, y in zip(a.adjoint_backward(seed), b.adjoint_backward(seed)):
        assert np.array_equal(x, y)
    a.close()
    b.close()
