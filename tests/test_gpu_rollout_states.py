"""The rollout's backward pass over the kept states of its forward pass against
the one that recomputes them from checkpoints: the same frames and gradients,
bit for bit, also when the backward pass runs twice; and the batched rollout's
block-tile forward and both of its reverse band heights against the per-grid
path, bit for bit."""
import numpy as np
import pytest
import torch

from cardiax_amd import adjoint
from cardiax_amd import params as P
from cardiax_amd import workloads as wl
from cardiax_amd.solve import State
from cardiax_amd.stimulus import Protocol

pytestmark = pytest.mark.gpu


def _problem(shape, seed):
    rng = np.random.default_rng(seed)
    f = np.zeros(shape, np.float32); f[:, : max(1, shape[1] // 10)] = 20.0
    st = State(*(torch.from_numpy(x.astype(np.float32)).cuda() for x in
                 (rng.uniform(0.3, 1.0, shape), rng.uniform(0.3, 1.0, shape),
                  rng.uniform(0.0, 1.0, shape))))
    D = torch.from_numpy(wl.scar_map(shape, rng)).cuda()
    return st, D, [(Protocol(3, 2, 11), torch.from_numpy(f).cuda())]


@pytest.mark.parametrize("shape,n,fe", [((3, 3), 1, 1), ((40, 52), 30, 7), ((64, 130), 31, 31),
                                        ((33, 65), 6, 10), ((120, 70), 0, 3)])
def test_kept_states_equal_recomputed(gpu, shape, n, fe, monkeypatch):
    st, D0, stims = _problem(shape, n)
    prm = P.PARAMSET_3

    def run(keep, every):
        monkeypatch.setattr(adjoint, "KEEP_BYTES", keep)
        D = D0.clone().requires_grad_(True)
        td = torch.tensor(prm.tau_d, device=gpu, requires_grad=True)
        fr = adjoint.rollout(D, td, prm.tau_r, prm.tau_si, st, prm, stims, 2, n, fe, 0.01, 0.01,
                             checkpoint_every=every)
        g = torch.linspace(0.5, 1.5, max(1, fr.numel()), device=gpu)[: fr.numel()].view_as(fr)
        first = torch.autograd.grad((fr * g).sum(), (D, td), retain_graph=True)
        second = torch.autograd.grad((fr * g).sum(), (D, td))
        assert all(torch.equal(a, b) for a, b in zip(first, second))
        return (fr.detach(),) + first

    kept = run(4 << 30, None)
    for other in (run(0, None), run(4 << 30, 4)):
        for a, b in zip(kept, other):
            assert torch.equal(a, b)


@pytest.mark.parametrize("shapes", [[(64, 64), (3, 5)], [(130, 200), (257, 111), (90, 64)],
                                    [(512, 400)] * 6 + [(300, 512)] * 4])
def test_batched_rollout_equals_per_grid(gpu, shapes):
    n, fe = 13, 4
    prm = P.PARAMSET_3
    probs = [_problem(sh, k) for k, sh in enumerate(shapes)]
    plan = adjoint.RolloutBatch([(st, prm, stims, 1.0)
                                 for st, _, stims in probs], n, fe, 0.01, 0.01,
                                checkpoint_every=5)
    Ds = [D.clone().requires_grad_(True) for _, D, _ in probs]
    frames = adjoint.rollout_batch(plan, Ds)
    grads = torch.autograd.grad(sum((f * f).sum() for f in frames), Ds)
    for (st, D0, stims), f, g in zip(probs, frames, grads):
        D = D0.clone().requires_grad_(True)
        fr = adjoint.rollout(D, prm.tau_d, prm.tau_r, prm.tau_si, st, prm, stims, 1.0, n, fe, 0.01,
                             0.01)
        assert torch.equal(f, fr)
        assert torch.equal(g, torch.autograd.grad((fr * fr).sum(), D)[0])
