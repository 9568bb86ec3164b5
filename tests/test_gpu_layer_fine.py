"""GetLayer at output sizes around the number of nodes from which the layer is
resampled on the host (2 for one of the layer), against a numpy gather of
the state before the last step (exact)."""
import pytest

from test_gpu_readback import test_get_layer_gathers_the_previous_state as _gathers

pytestmark = pytest.mark.gpu


# a 9 x 8 x 11 layer: twice its nodes, a few more, and many more
@pytest.mark.parametrize("outside", [False, True])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("out", [(9, 8, 22), (9, 16, 11), (9, 8, 23), (9, 8, 44), (36, 8, 11), (37, 8, 11),
                                 (50, 3, 60)])
def test_sizes(dtype, out, outside):
    _gathers(dtype, out, outside)
