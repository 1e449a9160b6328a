"""Block tiles of a batch against each simulation's own solve on the one-step
streaming kernel, bit for bit: batches of few tiles (4 steps per launch) and of
many (2 steps), sizes that the "t8" and "t16" options do not cover, step counts
that end a launch or a recorded graph early, stimuli on every step of a launch."""
import numpy as np
import pytest
import torch

from cardiax_amd import params as P
from cardiax_amd import workloads as wl
from cardiax_amd.batch import Batch, BatchSim
from cardiax_amd.stimulus import Protocol

from test_gpu_batch import _per_sim_variant

pytestmark = pytest.mark.gpu

SHAPES = {"few": [(64, 64), (48, 56), (113, 110), (96, 104)],
          "any": [(3, 3), (8, 300), (100, 100), (33, 65), (257, 40)],
          "many": [(300, 290), (256, 256), (400, 211), (64, 700)] * 4}


def _sims(shapes, seed):
    rng = np.random.default_rng(seed)
    names = sorted(P.ALL_PARAMSETS)
    out = []
    for k, sh in enumerate(shapes):
        f1 = np.zeros(sh, np.float32); f1[:, : max(1, sh[1] // 10)] = 20.0
        f2 = np.zeros(sh, np.float32); f2[sh[0] // 2:, sh[1] // 2:] = -3.0
        stims = [(Protocol(k % 5, 2, 1e9), f1), (Protocol(1, 3, 7), f2)][: 1 + k % 2]
        st = tuple(torch.from_numpy(x.astype(np.float32)).cuda() for x in
                   (rng.uniform(0.3, 1.0, sh), rng.uniform(0.3, 1.0, sh),
                    rng.uniform(0.0, 1.0, sh)))
        out.append(BatchSim(st, P.ALL_PARAMSETS[names[(3 * k) % len(names)]],
                            wl.scar_map(sh, rng), stims, float(k % 3), 0.01, 0.01))
    return out


@pytest.mark.parametrize("kind", sorted(SHAPES))
@pytest.mark.parametrize("option", [None, 8, 16])
@pytest.mark.parametrize("n", [1, 31, 67])
def test_block_tiles_equal_per_simulation_runs(gpu, kind, option, n):
    sims = _sims(SHAPES[kind], seed=n)
    refs = _per_sim_variant(sims, n, "stream2")
    with Batch(sims) as b:
        if option is not None:
            if kind == "any":
                with pytest.raises(NotImplementedError):
                    b.set_rows(option, two_step=True)
                return
            b.set_rows(option, two_step=True)
        b.run(n, use_graph=n != 31)
        torch.cuda.synchronize()
        for got, ref in zip(b.states, refs):
            for a, r in zip(got, ref):
                assert torch.equal(a, r)


def test_tuned_batch_that_no_block_option_covers(gpu):
    sims = _sims(SHAPES["any"], seed=9)
    refs = _per_sim_variant(sims, 40, "stream2")
    with Batch(sims) as b:
        res = b.autotune(n_steps=12)
        assert set(res["times_ms"]) == {"2", "4", "8", "16"} and not res["two_step"]
        b.run(40)
        torch.cuda.synchronize()
        for got, ref in zip(b.states, refs):
            for a, r in zip(got, ref):
                assert torch.equal(a, r)
