"""Which kernels the blur takes for outer products: one whose taps are off by 2^-47
of themselves keeps them, shown on an image where everything else cancels."""
import numpy as np
import pytest
import torch

from cardiax_amd import scars

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


@pytest.mark.parametrize("side", [3, 7, 8, 9])
def test_sides_around_the_rule(gpu, side):
    """Below and above the 64 taps up to which the bound on a tap grows, a kernel that is an outer product and one that is
    not, against float64: at most 81 products of values below 1, within 2^-24 of
    the result's rounding and 2^-46 of the sum."""
    rng = np.random.default_rng(side)
    img = rng.uniform(size=(37, 45)).astype(np.float32)
    for k in (scars.gauss_kernel(side, 2.0), rng.uniform(size=(side, side))):
        out = scars.convolve_same(torch.from_numpy(img).to(gpu), k).cpu().numpy()
        pad = np.pad(img.astype(np.float64), side)
        ref = np.zeros(img.shape)
        o = (side - 1) // 2
        for p in range(side):
            for q in range(side):
                i, j = side + o - p, side + o - q
                ref += k[p, q] * pad[i:i + img.shape[0], j:j + img.shape[1]]
        assert np.abs(out - ref).max() <= (2.0 ** -24 + 2.0 ** -46) * np.abs(ref).max()
