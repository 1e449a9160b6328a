"""Block tiles in their order over the dies: tile counts that 8 does not
divide, fewer bands than a group of 8, a last group of one band, one strip
only, and several rounds of the CUs; against the one-step streaming kernel, bit
for bit."""
import pytest
import torch

from cardiax_amd import params as P

from test_gpu_two_step import _inputs, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["tb64x2", "tb64x4", "tb32x2", "tb32x4"])
@pytest.mark.parametrize("shape", [(64, 102), (65, 103), (112, 62), (113, 620), (220, 150),
                                   (1500, 50), (40, 1700), (650, 613)])
def test_every_tile_once(gpu, variant, shape):
    st, D, stims = _inputs(shape, seed=shape[1])
    ref = _run("stream2", st, 1, 8, P.PARAMSET_3, D, stims)
    got = _run(variant, st, 1, 8, P.PARAMSET_3, D, stims)
    for name, a, b in zip("vwu", got, ref):
        assert torch.equal(a, b), (variant, shape, name)
