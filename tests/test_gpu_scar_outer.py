"""Which kernels the blur takes for outer products: one whose taps are off by 2^-47
of themselves keeps them, shown on an image where everything else cancels."""
import numpy as np
import pytest
import torch

from cardiax_amd import scars
from oracle import scar_oracle as so

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 13, 40])
def test_taps_are_kept(gpu, n):
    """Rows of alternating sign and an even number of equal tap rows cancel, which
    leaves the deviation. Every partial sum is a multiple of 2^-47 below 64 (at
    most 2 n terms of 1 are not yet cancelled), exact in double; so is the result
    in float32."""
    assert n <= 40
    k = np.ones((8, n))
    k[::2, n // 2:] += 2.0 ** -47
    img = torch.ones((50, 90), device=gpu)
    img[1::2] = -1.0
    out = scars.convolve_same(img, k).cpu().numpy()
    sign = np.ones((50, 1), np.float32)
    sign[1::2] = -1.0
    # the tap row p meets row i + 3 - p: even p meets the rows of the other parity
    expect = -sign * np.float32(2.0 ** -47 * 4 * (n - n // 2))
    inner = (slice(8, 42), slice(n, 90 - n) if n < 40 else slice(40, 50))
    assert np.array_equal(out[inner], np.broadcast_to(expect, out.shape)[inner])


@pytest.mark.parametrize("kh,kw", [(3, 3), (9, 9), (2, 24), (3, 11), (3, 12), (10, 8), (60, 2)])
def test_around_the_rule(gpu, kh, kw):
    """Kernels below and above the size from which an outer product runs as passes,
    one that is one and one that is not, against float64: the result's rounding and
    at most 264 double roundings (2^-44 of the sum)."""
    rng = np.random.default_rng(kh)
    img = rng.uniform(size=(37, 45)).astype(np.float32)
    for k in (np.outer(rng.uniform(0.5, 1.5, kh), rng.uniform(0.5, 1.5, kw)),
              rng.uniform(size=(kh, kw))):
        out = scars.convolve_same(torch.from_numpy(img).to(gpu), k).cpu().numpy()
        ref = so.convolve_same(img, k)
        assert np.abs(out - ref).max() <= (2.0 ** -23 + 2.0 ** -44) * np.abs(ref).max()


@pytest.mark.parametrize("kh,kw", [(3, 3), (6, 9), (17, 6), (30, 20)])
@pytest.mark.parametrize("outer", [True, False])
def test_non_finite_values_stay_in_their_windows(gpu, kh, kw, outer):
    rng = np.random.default_rng(kw)
    img = rng.uniform(size=(70, 80)).astype(np.float32)
    img[0, 3], img[35, 40], img[60, 79] = -np.inf, np.nan, np.inf
    k = (np.outer(rng.uniform(0.5, 1.5, kh), rng.uniform(0.5, 1.5, kw)) if outer
         else rng.uniform(0.1, 1.0, size=(kh, kw)))
    got = scars.convolve_same(torch.from_numpy(img).to(gpu), k).cpu().numpy()
    np.testing.assert_allclose(got, so.convolve_same(img, k), rtol=2 ** -22, atol=0)
