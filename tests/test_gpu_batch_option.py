"""The work-list option that a batch reports is the one it runs: before tuning,
after it (also where the tuner keeps block tiles that the sizes do not offer),
and pinned."""
import pytest
import torch

from cardiax_amd.batch import BATCH_OPTIONS, Batch

from test_gpu_batch_blocks import SHAPES, _sims

pytestmark = pytest.mark.gpu


def _tiles(option, shapes):
    """Tiles of a one-step option: bands of its rows by strips of 56 columns."""
    rows = int(option)
    return sum(-(-h // rows) * -(-w // 56) for h, w in shapes)


@pytest.mark.parametrize("kind", ["few", "any"])
def test_option_in_use(gpu, kind):
    with Batch(_sims(SHAPES[kind], seed=1)) as b:
        assert (b.option, b.steps_per_launch) == ("t8", 4)  # few tiles: 32 rows, 4 steps
        untuned = b.n_tiles
        res = b.autotune(n_steps=12)
        assert res["option"] == b.option
        offered = set(res["times_ms"])
        fastest = ("t" if res["two_step"] else "") + str(res["rows"])
        assert fastest in offered
        # the fastest offered option, or the untuned one in its place
        assert b.option in (fastest, "t8")
        if b.option == "t8":
            assert b.n_tiles == untuned
        for rows in (2, 4, 8, 16):
            b.set_rows(rows)
            assert (b.option, b.steps_per_launch) == (str(rows), 1)
            assert b.n_tiles == _tiles(b.option, SHAPES[kind])
        b.run(3)
        torch.cuda.synchronize()
    with pytest.raises(RuntimeError):
        b.option


def test_steps_of_the_block_options(gpu):
    with Batch(_sims(SHAPES["many"], seed=2)) as b:
        steps = {}
        for rows in (8, 16):
            b.set_rows(rows, two_step=True)
            assert b.option == "t%d" % rows and b.option in BATCH_OPTIONS
            steps[b.option] = b.steps_per_launch
        assert steps == {"t8": 2, "t16": 3}
