"""Host logic only: the kernel that a solve of several steps and a single step of
a shape run, as the library reports it. The launches take the same functions."""
import pytest

from cardiax_amd import _lib, autotune

BLOCKS = ("tb64x2", "tb64x4", "tb32x2", "tb32x4")


@pytest.fixture
def variant():
    L = _lib.lib()
    prev = L.fk_set_forward_variant(0)
    yield lambda name: L.fk_set_forward_variant(_lib.VARIANTS[name])
    L.fk_set_forward_variant(prev)


@pytest.mark.parametrize("shape,solve", [
    ((3, 3), "tb32x4"), ((128, 128), "tb32x4"),       # 32 rows, 4 steps
    ((500, 500), "tb64x4"), ((4096, 4096), "tb64x4"),  # 48 rows, 3 steps
    ((700, 600), "tb32x2"),                            # 64 rows, 3 steps
    ((2048, 2048), "tb64x2"),                          # 32 rows, 2 steps
    ((100000, 100), "tile16")])
def test_automatic_solves(variant, shape, solve):
    assert autotune.solve_variant(shape) == solve


@pytest.mark.parametrize("name,shape,solve,step", [
    ("auto", (1024, 1024), None, "stream2"), ("auto", (2048, 2048), None, "stream2"),
    ("auto", (40000, 100), None, "stream4"), ("auto", (100000, 100), "tile16", "tile16"),
    ("stream16", (64, 64), "stream16", "stream16"),
    ("streamc8", (64, 64), "streamc8", "stream8"), ("streamc2", (64, 64), "streamc2", "stream2"),
    ("pair2", (64, 64), "pair2", "pair2"), ("pair2", (64, 63), "stream2", "stream2"),
    ("pair4", (64, 63), "stream4", "stream4"),
    ("streamt12", (1024, 1024), "streamt12", "stream2"),
    ("streamt12", (39, 1024), "stream2", "stream2")])
def test_solves_and_single_steps(variant, name, shape, solve, step):
    variant(name)
    if solve is None:
        assert autotune.solve_variant(shape) in BLOCKS
    else:
        assert autotune.solve_variant(shape) == solve
    assert autotune.step_variant(shape) == step


def test_refused_grids(variant):
    for query in (autotune.solve_variant, autotune.step_variant):
        for shape in ((2, 64), (64, 2), ((1 << 18) + 1, 64)):
            with pytest.raises(ValueError):
                query(shape)


@pytest.mark.parametrize("name", BLOCKS)
def test_single_steps_of_block_variants(variant, name):
    """A shape whose tuned solve runs block tiles takes the 2-row bands for single
    steps, as the last step of such a solve does."""
    variant(name)
    assert autotune.solve_variant((1024, 1024)) == name
    assert autotune.step_variant((1024, 1024)) == "stream2"


def test_a_launch_stays_below_2_32_threads(variant):
    """1024 threads per 8 x 32 cells of a 32-row tile of 4 steps: above 1.07e9 cells
    they would exceed what a launch may hold."""
    variant("tb32x4")
    assert autotune.solve_variant((32768, 32000)) == "tb32x4"  # 4.19e9 threads
    assert autotune.solve_variant((32768, 33000)) == "tb64x4"
    assert autotune.solve_variant((1 << 18, 8192)) == "tb64x4"
