"""Memory of the states that a rollout keeps for its backward pass: given back
with the graph, also while the frames and the loss are held, and bounded over
all rollouts that await their backward pass."""
import pytest
import torch
import torch.utils.checkpoint

from cardiax_amd import adjoint
from cardiax_amd import params as P

from test_gpu_rollout_states import _problem

pytestmark = pytest.mark.gpu

SHAPE, N, FE, PRM = (256, 240), 60, 20, P.PARAMSET_3
STATES = 12 * (N + 1) * SHAPE[0] * SHAPE[1]


def _rollout(seed):
    st, D, stims = _problem(SHAPE, seed)
    D.requires_grad_(True)
    fr = adjoint.rollout(D, PRM.tau_d, PRM.tau_r, PRM.tau_si, st, PRM, stims, 1, N, FE, 0.01,
                         0.01)
    return D, fr, (fr * fr).sum()


def test_given_back_with_the_graph(gpu):
    before = torch.cuda.memory_allocated()
    D, fr, loss = _rollout(1)
    assert torch.cuda.memory_allocated() - before >= STATES
    loss.backward()
    # what is left: D, its gradient, the frames and the problem's own fields
    assert torch.cuda.memory_allocated() - before < STATES / 4
    with pytest.raises(RuntimeError, match="second time"):
        loss.backward()


def test_bounded_over_live_rollouts(gpu, monkeypatch):
    monkeypatch.setattr(adjoint, "KEEP_BYTES", 5 * STATES // 2)
    before = torch.cuda.memory_allocated()
    runs = [_rollout(k) for k in range(5)]
    # two trajectories, and checkpoints every 8 steps for the other three
    assert torch.cuda.memory_allocated() - before < 4 * STATES
    torch.autograd.backward([r[2] for r in runs])
    grads = [r[0].grad for r in runs]
    del runs
    monkeypatch.setattr(adjoint, "KEEP_BYTES", 0)
    for k, g in enumerate(grads):
        D, _, loss = _rollout(k)
        loss.backward()
        assert torch.equal(g, D.grad)
    monkeypatch.setattr(adjoint, "KEEP_BYTES", 3 * STATES // 2)
    held = []
    for k in range(3):  # one after another they all keep theirs
        before = torch.cuda.memory_allocated()
        held.append(_rollout(k))
        assert torch.cuda.memory_allocated() - before >= STATES
        held[-1][2].backward()


def test_not_kept_under_saved_tensor_hooks(gpu):
    D, _, loss = _rollout(2)
    loss.backward()
    ref = D.grad
    before = torch.cuda.memory_allocated()
    with torch.autograd.graph.save_on_cpu():
        D, fr, loss = _rollout(2)
        assert torch.cuda.memory_allocated() - before < STATES
    loss.backward()
    assert torch.equal(D.grad, ref)
    st, D, stims = _problem(SHAPE, 2)
    D.requires_grad_(True)
    fr = torch.utils.checkpoint.checkpoint(
        lambda d: adjoint.rollout(d, PRM.tau_d, PRM.tau_r, PRM.tau_si, st, PRM, stims, 1, N, FE,
                                  0.01, 0.01), D, use_reentrant=False)
    (fr * fr).sum().backward()
    assert torch.equal(D.grad, ref)
