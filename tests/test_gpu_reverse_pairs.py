"""The reverse step of bands of 2 rows on one grid, above 2048 of them: one step
against FP64 autograd (D, state and taus), and rollouts against the batched bands
of 2 and 4 rows, bit for bit, tau gradients included."""
import pytest
import torch

from cardiax_amd import adjoint
from cardiax_amd import params as P

from test_gpu_adjoint import test_single_step_vjp_matches_autograd as _vjp
from test_gpu_rollout_states import _problem

pytestmark = pytest.mark.gpu

LARGE = [(250, 918), (249, 919), (1031, 220)]  # odd and even heights, 5 to 18 strips


@pytest.mark.parametrize("shape", LARGE)
@pytest.mark.parametrize("pname", ["3", "2"])
def test_one_step(gpu, shape, pname):
    """Reference and tolerance of the single-step test (FP64 autograd, 2e-5 of the
    largest value, 1e-4 for a tau)."""
    _vjp(gpu, shape, pname)


def _batched(probs, n, fe):
    prm = P.PARAMSET_3
    with adjoint.RolloutBatch([(st, prm, stims, 1.0) for st, _, stims in probs], n, fe, 0.01,
                              0.01) as plan:
        frames = [f.clone() for f in plan.forward([D for _, D, _ in probs])]
        gD, gt = plan.backward([2.0 * f for f in frames], tau_grads=True)
        return frames, [g.clone() for g in gD], gt.clone()


@pytest.mark.parametrize("shape", LARGE)
def test_rollout_equals_batched_bands(gpu, shape):
    n, fe, prm = 9, 3, P.PARAMSET_3
    prob = _problem(shape, 5)
    st, D0, stims = prob
    D = D0.clone().requires_grad_(True)
    taus = [torch.tensor(float(x), device=gpu, requires_grad=True)
            for x in (prm.tau_d, prm.tau_r, prm.tau_si)]
    fr = adjoint.rollout(D, *taus, st, prm, stims, 1.0, n, fe, 0.01, 0.01)
    gD, *gt = torch.autograd.grad((fr * fr).sum(), [D] + taus)
    fours = [_problem((512, 500), k) for k in range(6)]
    for extra in ([], fours):  # bands of 2 rows, of 4
        frames, grads, tau = _batched([prob] + extra, n, fe)
        assert torch.equal(frames[0], fr)
        assert torch.equal(grads[0], gD)
        for f in range(3):
            assert torch.equal(tau[0, f], gt[f]), f


def test_small_grids_keep_their_tau_gradients(gpu):
    """A wave per row, bands of 2 and of 4: the same sums."""
    small = [_problem(sh, k) for k, sh in enumerate([(3, 3), (27, 55), (40, 109), (101, 70)])]
    ref = _batched(small, 6, 3)[2]
    for fill in (2, 6):
        got = _batched(small + [_problem((512, 500), k) for k in range(fill)], 6, 3)[2]
        assert torch.isfinite(ref).all() and torch.equal(got[: len(small)], ref)
