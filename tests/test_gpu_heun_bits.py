"""Heun steps do not depend on the tiling, bit for bit: a corner of a large grid
solved by itself agrees with the large solve wherever the cut is out of reach, at
sizes that take each of the tilings; solves agree with single steps; and one step
is within half a rounding per stage of its definition."""
import pytest
import torch

from cardiax_amd import params as P
from cardiax_amd import solve

from test_gpu_two_step import _inputs

pytestmark = pytest.mark.gpu

LARGE = (3000, 2000)  # 40 rows, 1 step
CORNERS = [(150, 170),   # 32 rows, 2 steps
           (517, 389),   # 48 rows, 2 steps
           (760, 761),   # 64 rows, 1 step
           (1201, 1203)]
DT, DX, PRM = 0.01, 0.01, P.PARAMSET_3


def _problem(gpu):
    st, D, stims = _inputs(LARGE, seed=9)
    return st, torch.from_numpy(D).to(gpu), [(s[0], torch.as_tensor(s[1]).to(gpu)) for s in stims]


@pytest.mark.parametrize("steps", [1, 2, 3])
def test_corners_of_a_large_grid(gpu, steps):
    st, D, stims = _problem(gpu)
    full = solve._forward_heun(st, 3, 3 + steps, PRM, D, stims, DT, DX)
    reach = 10 * steps  # two stages of at most 5 cells
    for h, w in CORNERS:
        for rows, cols, keep in (
                (slice(0, h), slice(0, w), (slice(0, h - reach), slice(0, w - reach))),
                (slice(-h, None), slice(-w, None), (slice(reach, h), slice(reach, w)))):
            cut = lambda x: x[rows, cols].contiguous()
            got = solve._forward_heun(tuple(cut(x) for x in st), 3, 3 + steps, PRM, cut(D),
                                      [(p, cut(f)) for p, f in stims], DT, DX)
            for a, b in zip(got, full):
                assert torch.isfinite(a).all()
                assert torch.equal(a[keep], cut(b)[keep]), (h, w, steps)


@pytest.mark.parametrize("shape", CORNERS + [(3, 3), (33, 64), (640, 650)])
def test_solves_equal_single_steps(gpu, shape):
    st, D, stims = _inputs(shape, seed=shape[0])
    D = torch.from_numpy(D).to(gpu)
    stims = [(s[0], torch.as_tensor(s[1]).to(gpu)) for s in stims]
    x = solve.State(*st)
    for t in range(2, 7):
        x = solve.step_heun(x, t, PRM, D, stims, DT, DX)
    for a, b in zip(solve._forward_heun(st, 2, 7, PRM, D, stims, DT, DX), x):
        assert torch.equal(a, b)


@pytest.mark.parametrize("shape", CORNERS + [(3, 3), (20, 63), (65, 111)])
def test_one_step_of_its_definition(gpu, shape):
    """x + dt k1 and x + (k1 + k2) dt / 2 from single evaluations of the right-hand
    side in float64, rounded once a stage: half a unit in the last place of values
    below 2 (1.2e-7) in either, the first through dynamics that amplify it by less
    than 2 per stage: 4 x 1.2e-7."""
    st, D, stims = _inputs(shape, seed=1 + shape[0])
    D = torch.from_numpy(D).to(gpu)
    stims = [(s[0], torch.as_tensor(s[1]).to(gpu)) for s in stims]
    dt = float(torch.tensor(DT, dtype=torch.float32))
    got = solve.step_heun(st, 4, PRM, D, stims, DT, DX)
    k1 = solve.step(st, 4, PRM, D, stims, DX)
    x1 = solve.State(*((a.double() + dt * k.double()).float() for a, k in zip(st, k1)))
    k2 = solve.step(x1, 4, PRM, D, stims, DX)
    for a, x, k, q in zip(got, st, k1, k2):
        ref = x.double() + (k + q).double() * (0.5 * dt)
        assert (a.double() - ref).abs().max().item() <= 4 * 1.2e-7
