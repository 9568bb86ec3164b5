"""Z lines whose length is no multiple of a lane's rows or of 16 bytes: the Z
sweep and the transposed Z solve read them in unaligned vectors, the last run
of a line reaching past its end.  Against the oracle, with the bars of the
other parity tests (1e-11 in FP64, 1e-5 in FP32, gradients 1e-9)."""
import numpy as np
import pytest

import adjoint_cases as ac
from cmcx import domains
from cmcx.solver import make_solver
from gpu_util import rel_l2, say
from test_gpu_adjoint import EVERY, STEPS, _oracle_grads
from test_gpu_batch import _check_batch
from test_gpu_edges import FUSED, _compare, _long

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,nz", [("f32", n) for n in (3, 31, 33, 63, 66, 127, 129, 187, 255, 257, 511)] +
                         [("f64", n) for n in (3, 33, 63, 67, 129, 187, 255)])
def test_ragged_z_lines(dtype, nz):
    say(f"[ragged z] {dtype} nz={nz}")
    _compare(_long((7, 6, nz), nz), dtype, FUSED, [(0, 0, z) for z in range(8)])


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_ragged_batch(dtype):
    """Short lines beside long ones: lanes sized for the longest line (8 rows)
    over a grid of 3 x 3 x 3 nodes, last in memory, and odd boxes."""
    rng = np.random.default_rng(3)
    doms = [domains.random_domain(s, rng, 0.1) for s in ((6, 5, 201), (9, 8, 17), (5, 7, 66), (3, 3, 3))]
    say(f"[ragged batch] {dtype}")
    _check_batch(doms, dtype, FUSED, steps=2)


@pytest.mark.parametrize("nz", [3, 35, 67, 131])
def test_ragged_adjoint(nz):
    rng = np.random.default_rng(nz)
    d = domains.random_domain((9, 8, nz), rng, 0.08, free_faces=True)
    d.re, d.dt = 50.0, ac.DT
    seed = rng.normal(size=(4, d.n)) * (d.type == domains.NODE_IN)
    ogb, ocb, opb = _oracle_grads(d, seed)
    s = make_solver(d, "f64", path=FUSED)
    s.adjoint_forward(STEPS, ac.DT, ac.G, EVERY)
    gb, sb, pb = s.adjoint_backward(seed)
    say(f"[ragged adjoint] nz={nz}: node values {rel_l2(gb, ogb):.2e}, initial state {rel_l2(sb, ocb):.2e}")
    assert rel_l2(gb, ogb) < 1e-9 and rel_l2(sb, ocb) < 1e-9
    assert np.allclose(pb, opb, rtol=1e-9, atol=0)
    s.close()
