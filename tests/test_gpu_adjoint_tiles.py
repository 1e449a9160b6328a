"""The reverse step at the sizes where its tiles change: axes shorter than the
edge tables, the smallest ones with central cells, one column and one row past
a strip (54 columns) and a band, an odd last row. Reference and tolerance are
those of the single-step test (FP64 autograd, 2e-5 of the largest value)."""
import pytest

from test_gpu_adjoint import test_single_step_vjp_matches_autograd as _vjp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 3), (4, 54), (8, 55), (13, 26), (16, 27), (17, 53),
                                   (26, 108), (27, 109), (28, 59), (31, 121), (55, 28)])
@pytest.mark.parametrize("pname", ["3", "2"])
def test_tiles(gpu, shape, pname):
    _vjp(gpu, shape, pname)
