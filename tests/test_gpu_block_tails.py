"""Solves whose steps do not fill the launches of a 3-step tiling, on a grid whose
fields exceed the 256 MB cache: the bits of single steps, and no slower than two
steps per launch on streaming bands."""
import pytest
import torch

from cardiax_amd import _lib, autotune, solve
from cardiax_amd.params import PARAMSET_3

from test_gpu_two_step import _inputs, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 2, 4, 5, 6, 7])
def test_equal_single_steps(gpu, steps):
    shape = (3001, 3300)
    assert autotune.solve_variant(shape) == "tb64x4"  # 48 rows, 3 steps
    st, D, stims = _inputs(shape, seed=steps)
    ref = _run("stream2", st, 3, 3 + steps, PARAMSET_3, D, stims)
    got = _run("auto", st, 3, 3 + steps, PARAMSET_3, D, stims)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("steps", [2, 4])
def test_short_solves_are_no_slower(gpu, steps):
    shape = (4096, 4096)
    D = torch.full(shape, 1e-3, device=gpu)
    st = solve.State(*(torch.full(shape, x, device=gpu) for x in (0.9, 0.8, 0.3)))
    L, best = _lib.lib(), {}
    for _ in range(12):
        for name in ("auto", "streamt16"):
            prev = L.fk_set_forward_variant(_lib.VARIANTS[name])
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            solve._forward_euler(st, 0, steps, PARAMSET_3, D, [], 0.01, 0.01)
            e[1].record()
            e[1].synchronize()
            L.fk_set_forward_variant(prev)
            best[name] = min(best.get(name, 1e9), e[0].elapsed_time(e[1]))
    assert best["auto"] < 1.1 * best["streamt16"]
