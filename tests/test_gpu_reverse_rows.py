"""The reverse step with a wave per row, with bands of 2 rows and of 4: a plan
whose other problems move it from one to the next keeps each problem's frames and
gradients bit for bit, at odd and even heights and one-strip and many-strip
widths."""
import pytest
import torch

from cardiax_amd import adjoint
from cardiax_amd import params as P

from test_gpu_rollout_states import _problem

pytestmark = pytest.mark.gpu

SMALL = [(3, 3), (4, 54), (27, 55), (40, 109), (101, 70)]
FILL = {"rows": [], "pairs": [(512, 500)] * 2, "fours": [(512, 500)] * 6}


@pytest.mark.parametrize("fill", ["pairs", "fours"])
def test_band_heights_agree(gpu, fill):
    n, fe, prm = 9, 3, P.PARAMSET_3

    def run(extra):
        probs = [_problem(sh, k) for k, sh in enumerate(SMALL + extra)]
        plan = adjoint.RolloutBatch([(st, prm, stims, 1.0) for st, _, stims in probs], n, fe,
                                    0.01, 0.01)
        Ds = [D.clone().requires_grad_(True) for _, D, _ in probs]
        frames = adjoint.rollout_batch(plan, Ds)
        grads = torch.autograd.grad(sum((f * f).sum() for f in frames), Ds)
        return frames[: len(SMALL)], grads[: len(SMALL)]

    one, other = run(FILL["rows"]), run(FILL[fill])
    for a, b in zip(one[0] + one[1], other[0] + other[1]):
        assert torch.isfinite(a).all()
        assert torch.equal(a, b)
