"""Results read back: GetLayer's device resampling against a numpy gather of
the state before the last step (exact), and fields_device into program buffers
at any element offset against fields() (exact)."""
import numpy as np
import pytest
import torch

from cmcx import domains
from cmcx.solver import make_batch, make_solver
from gpu_util import say

pytestmark = pytest.mark.gpu

NP = {"f32": np.float32, "f64": np.float64}


def _grid(shape, seed, outside):
    d = domains.random_domain(shape, np.random.default_rng(seed), 0.1)
    if outside:  # a slab of outside nodes behind a wall
        t = d.type.reshape(shape)
        t[:2] = domains.NODE_OUT
        t[2] = domains.NODE_BOUND
    d.dt = 1e-3
    return d


@pytest.mark.parametrize("outside", [False, True])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("out", [(0, 0, 0), (1, 1, 1), (6, 0, 17), (7, 5, 4), (31, 40, 29), (110, 101, 103)])
def test_get_layer_gathers_the_previous_state(dtype, out, outside):
    """The last size spans two device chunks of 2^20 nodes."""
    d = _grid((9, 8, 11), 5, outside)
    s = make_solver(d, dtype, path=1)
    say(f"[get_layer] {dtype} out={out} outside={outside}")
    for k in range(3):
        s.UpdateBoundaries()
        f = s.fields()
        s.TimeStep(d.dt, 2, 1, False)
        vel, T = s.GetLayer(*out)
        at = [np.arange(o or n) * n // (o or n) for o, n in zip(out, d.shape)]
        gone = (d.type == domains.NODE_OUT).reshape(d.shape)
        want = [np.where(gone, NP[dtype](99999), f[i].reshape(d.shape))[np.ix_(*at)].ravel() for i in (0, 1, 2, 4)]
        assert np.array_equal(vel, np.stack(want[:3], 1)), k
        assert np.array_equal(T, want[3].astype(np.float64)), k
    s.close()


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_fields_device_any_offset(dtype, shift):
    """Odd node counts, buffers that start off a 16-byte boundary, some absent,
    and a batch whose grids lie back to back in the program's arrays."""
    ds = [_grid(s, i, False) for i, s in enumerate([(5, 7, 9), (3, 3, 3), (8, 6, 10)])]
    s = make_batch(ds, dtype)
    s.run(2, 1e-3, 2, 1)
    n = sum(d.n for d in ds)
    ty = torch.float32 if dtype == "f32" else torch.float64
    say(f"[fields_device] {dtype} shift={shift}")
    buf = torch.full((5, n + shift + 1), -7.0, dtype=ty, device="cuda")
    o = shift
    for i, d in enumerate(ds):
        s.select(i)
        ptrs = [buf[k, o:o + d.n].data_ptr() for k in range(5)]
        if i == 1:
            ptrs[1] = ptrs[3] = None
        s.fields_device(*ptrs)
        for k, f in enumerate(s.fields()):
            got = buf[k, o:o + d.n].cpu().numpy()
            want = np.full(d.n, -7.0, NP[dtype]) if i == 1 and k in (1, 3) else f
            assert np.array_equal(got, want), (i, k)
        o += d.n
    assert (buf[:, :shift] == -7).all() and (buf[:, o:] == -7).all()
    s.close()
