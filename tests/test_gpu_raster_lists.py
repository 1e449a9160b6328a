"""The rasteriser's crossing lists against the brute-force oracle, bit for bit:
more polygons than one pass holds, more crossings than a list holds, and the
widths around a wave."""
import numpy as np
import pytest

from cardiax_amd import scars
from oracle import scar_oracle as so

pytestmark = pytest.mark.gpu


def _comb(n, shape):
    """A closed zigzag whose middle rows cross n edges and more."""
    H, W = shape
    rows = np.where(np.arange(n) % 2 == 0, 0.3 * H, 0.8 * H)
    cols = np.linspace(1.0, W - 2.0, n)
    return (np.concatenate([rows, [0.9 * H, 0.9 * H]]),
            np.concatenate([cols, [W - 2.0, 1.0]]))


@pytest.mark.parametrize("n_polys", [1, 31, 32, 33, 70])
@pytest.mark.parametrize("shape", [(13, 64), (40, 65), (61, 200)])
def test_many_polygons(gpu, n_polys, shape):
    rng = np.random.default_rng(n_polys)
    cs = []
    for _ in range(n_polys):
        n = int(rng.integers(3, 90))
        th = np.sort(rng.uniform(0, 2 * np.pi, n))
        rad = rng.uniform(0.5, 6.0, n)
        cs.append((rng.uniform(0, shape[0]) + rad * np.sin(th),
                   rng.uniform(0, shape[1]) + rad * np.cos(th)))
    assert np.array_equal(scars.rasterize(cs, shape).cpu().numpy(), so.union_mask(cs, shape))


@pytest.mark.parametrize("n", [64, 255, 256, 257, 900])
def test_many_crossings(gpu, n):
    shape = (37, 301)
    small = ([3.0, 30.0, 12.0], [2.0, 40.0, 90.0])
    for cs in ([_comb(n, shape)], [small, _comb(n, shape), small]):
        assert np.array_equal(scars.rasterize(cs, shape).cpu().numpy(),
                              so.union_mask(cs, shape))
