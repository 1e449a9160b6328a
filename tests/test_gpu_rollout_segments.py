"""The batched rollout's forward and backward pass at the checkpoint intervals that
leave single steps over (every step alone, one after whole launches, one in the
last segment or in a recomputation), against the per-grid path, bit for bit."""
import pytest
import torch

from cardiax_amd import adjoint
from cardiax_amd import params as P

from test_gpu_rollout_states import _problem

pytestmark = pytest.mark.gpu

SHAPES = {"few": [(3, 3), (5, 60), (64, 113), (41, 57)],  # 4 steps per launch
          "many": [(300, 290), (256, 256), (400, 211)] * 4}  # 2 steps per launch


@pytest.mark.parametrize("kind", sorted(SHAPES))
@pytest.mark.parametrize("every", [1, 2, 3, 5, 6, 13])
def test_single_steps(gpu, kind, every):
    n, fe, prm = 13, 4, P.PARAMSET_3
    probs = [_problem(sh, k) for k, sh in enumerate(SHAPES[kind])]
    with adjoint.RolloutBatch([(st, prm, stims, 1.0) for st, _, stims in probs], n, fe, 0.01,
                              0.01, checkpoint_every=every) as plan:
        Ds = [D.clone().requires_grad_(True) for _, D, _ in probs]
        frames = adjoint.rollout_batch(plan, Ds)
        grads = torch.autograd.grad(sum((f * f).sum() for f in frames), Ds)
    for (st, D0, stims), f, g in zip(probs, frames, grads):
        D = D0.clone().requires_grad_(True)
        fr = adjoint.rollout(D, prm.tau_d, prm.tau_r, prm.tau_si, st, prm, stims, 1.0, n, fe,
                             0.01, 0.01)
        assert torch.equal(f, fr)
        assert torch.equal(g, torch.autograd.grad((fr * fr).sum(), D)[0])
