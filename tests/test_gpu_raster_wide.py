"""The rasteriser on images much wider than tall: the same mask as the oracle, and
the work spread over the columns as over the rows."""
import numpy as np
import pytest
import torch

from cardiax_amd import scars
from oracle import scar_oracle as so

pytestmark = pytest.mark.gpu


def _ellipses(shape, n=5):
    H, W = shape
    t = np.linspace(0.0, 2.0 * np.pi, 101)
    return [(H * (0.5 + 0.4 * np.sin(t)), W * (0.2 + 0.15 * k + 0.1 * np.cos(t)))
            for k in range(n)]


@pytest.mark.parametrize("shape", [(1, 255), (2, 256), (3, 257), (5, 513), (4, 3001)])
def test_wide_images(gpu, shape):
    cs = _ellipses(shape, 40)
    assert np.array_equal(scars.rasterize(cs, shape).cpu().numpy(), so.union_mask(cs, shape))


def _time(shape):
    cs, best = _ellipses(shape), float("inf")
    out = torch.empty(shape, device="cuda")
    for _ in range(30):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        scars.rasterize(cs, shape, out=out)
        e[1].record()
        e[1].synchronize()
        best = min(best, e[0].elapsed_time(e[1]))
    return best


def test_wide_images_fill_the_gpu(gpu):
    """As many pixels on 4 rows as on 640: a wave per row would take ten times as
    long."""
    assert _time((4, 102400)) < 4.0 * _time((640, 640))
