"""fields_device and the ends of a program's allocations: an array whose last node
is its allocation's last is written whole, one that ends before is refused, as the
runtime's copies refuse it, and nothing is written past it (the arrays here are
smaller than a page)."""
import ctypes

import numpy as np
import pytest

from cmcx import _lib, domains
from cmcx.solver import make_solver
from gpu_util import say
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


def _get(hip, p, n, ty):
    a = np.zeros(n, ty)
    assert hip.h.hipMemcpy(ctypes.c_void_p(a.ctypes.data), ctypes.c_void_p(p), a.nbytes, 2) == 0
    return a


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("short", [None, 0, 1, 2, 3])
def test_allocation_ends(dtype, short):
    hip = _Hip()
    d = domains.random_domain((6, 5, 7), np.random.default_rng(4), 0.1)
    s = make_solver(d, dtype, path=1)
    s.run(2, 1e-3, 2, 1)
    ty, n = s.np_dtype, d.n
    nb = n * np.dtype(ty).itemsize
    say(f"[device arrays] {dtype} short={short}")
    # u, v, w, p, T: each its own allocation, of exactly the grid's size
    at = [hip.alloc(nb) for _ in range(5)]
    if short is not None:
        k = (0, 1, 2, 4)[short]
        at[k] = hip.upload(np.zeros(n // 2, ty))
        with pytest.raises(_lib.CmcxError) as e:
            s.fields_device(*at)
        assert e.value.code == _lib.CMCX_ERR_HIP
        s.synchronize()
        assert not _get(hip, at[k], n // 2, ty).any()
        # the last element that fits starts the array: refused as well
        at[k] = hip.alloc(nb) + nb - np.dtype(ty).itemsize
        with pytest.raises(_lib.CmcxError):
            s.fields_device(*at)
    else:
        s.fields_device(*at)
        for p, f in zip(at, s.fields()):
            assert np.array_equal(_get(hip, p, n, ty), f)
        # one allocation for all, the last array to its end
        b = hip.alloc(5 * nb)
        s.fields_device(*[b + k * nb for k in range(5)])
        for k, f in enumerate(s.fields()):
            assert np.array_equal(_get(hip, b + k * nb, n, ty), f)
    s.close()
    hip.free()
