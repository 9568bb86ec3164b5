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
