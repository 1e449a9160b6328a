"""Gradients with respect to tau_d, tau_r and tau_si when neighbouring rows'
terms nearly cancel: the rows are added in double, so a small row next to two
large ones of opposite sign comes out whole. For the reverse step's wave per
row, bands of 2 rows and bands of 4, at even and odd heights."""
import math

import pytest
import torch

from cardiax_amd import adjoint
from cardiax_amd import params as P
from cardiax_amd.solve import State

pytestmark = pytest.mark.gpu

V, W_, U, DT, DX = 0.75, 0.875, 0.5, 0.01, 0.01


def _problem(shape, gpu):
    """A uniform state (no diffusion), and a cotangent of u after one step whose
    rows are 2^30, 1, -2^30, 1, ... : the large rows cancel exactly."""
    st = State(*(torch.full(shape, x, device=gpu) for x in (V, W_, U)))
    lam = torch.zeros(shape, device=gpu)
    n = shape[0] // 4 * 4
    for r, x in enumerate((2.0 ** 30, 1.0, -2.0 ** 30, 1.0)):
        lam[r:n:4] = x
    return st, torch.full(shape, 1e-3, device=gpu), lam, (n // 2) * shape[1]


def _expected(prm, weight):
    """dt x (d j_ion / d tau) x the sum of the small cotangents."""
    s = 0.5 * (1.0 + math.tanh(prm.k * (U - prm.V_csi)))
    assert U >= prm.V_c
    d = (-V * (U - prm.V_c) * (1.0 - U) / prm.tau_d ** 2, 1.0 / prm.tau_r ** 2,
         -W_ * s / prm.tau_si ** 2)
    return [DT * weight * x / prm.Cm for x in d]


def _check(got, prm, weight):
    """A term is a product of at most eight float32 factors, tanh among them
    within 2e-6; sums of 54 equal terms add 4e-6."""
    for g, e in zip(got, _expected(prm, weight)):
        assert float(g) == pytest.approx(e, rel=1e-5)


@pytest.mark.parametrize("shape", [(8, 60), (29, 117), (102, 64),  # a wave per row
                                   (520, 900), (521, 901)])  # above 2048 bands: 2 rows
def test_rollout(gpu, shape):
    prm = P.PARAMSET_3
    st, D, lam, weight = _problem(shape, gpu)
    taus = [torch.tensor(float(x), device=gpu, requires_grad=True)
            for x in (prm.tau_d, prm.tau_r, prm.tau_si)]
    fr = adjoint.rollout(D, *taus, st, prm, [], 0, 1, 1, DT, DX)
    _check(torch.autograd.grad(fr, taus, lam[None]), prm, weight)


@pytest.mark.parametrize("fill", [0, 2, 6])  # a wave per row, bands of 2 and of 4 rows
def test_rollout_batch(gpu, fill):
    prm = P.PARAMSET_3
    shapes = [(8, 60), (29, 117)] + [(512, 500)] * fill
    probs = [_problem(sh, gpu) for sh in shapes]
    with adjoint.RolloutBatch([(st, prm, [], 0) for st, _, _, _ in probs], 1, 1, DT, DX) as plan:
        plan.forward([D for _, D, _, _ in probs])
        _, gt = plan.backward([lam[None] for _, _, lam, _ in probs], tau_grads=True)
        for row, (_, _, _, weight) in zip(gt, probs):
            _check(row, prm, weight)
