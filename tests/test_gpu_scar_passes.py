"""The blur by passes (kernels that are an outer product) against scipy, at the
edges of its segments and spans, and the kernels that must not take it."""
import numpy as np
import pytest
import torch

from cardiax_amd import scars
from oracle import scar_oracle as so

pytestmark = pytest.mark.gpu


def _blur(img, k):
    return scars.convolve_same(torch.from_numpy(img).cuda(), k).cpu().numpy()


@pytest.mark.parametrize("H,W", [(1, 1), (5, 3), (7, 513), (33, 512), (130, 1100)])
@pytest.mark.parametrize("kh,kw", [(1, 1), (1, 9), (8, 1), (9, 24), (31, 250), (12, 300)])
def test_outer_product_kernels(gpu, H, W, kh, kw):
    rng = np.random.default_rng(H + 7 * kw)
    img = rng.uniform(size=(H, W)).astype(np.float32)
    k = np.outer(rng.uniform(0.5, 1.5, kh), rng.uniform(0.5, 1.5, kw))
    # double sums, one rounding to float32 (2^-24); the factors' product may
    # be 2^-46 off a tap
    np.testing.assert_allclose(_blur(img, k), so.convolve_same(img, k), rtol=2 ** -23, atol=0)


@pytest.mark.parametrize("case", ["cut", "centre0", "nan", "almost"])
def test_other_kernels_keep_every_tap(gpu, case):
    rng = np.random.default_rng(3)
    img = rng.uniform(size=(70, 90)).astype(np.float32)
    k = np.outer(rng.uniform(0.5, 1.5, 14), rng.uniform(0.5, 1.5, 11))
    if case == "cut":
        k = so.gauss_kernel(40, 1.5)  # its tail is zeroed
        assert (k == 0).any() and (k > 0).any()
    elif case == "centre0":
        k[6, :] = 0.0
    elif case == "nan":
        k[2, 3] = np.nan
    else:
        k[0, 0] *= 1 + 1e-6
    np.testing.assert_allclose(_blur(img, k), so.convolve_same(img, k), rtol=2 ** -23, atol=1e-9)
    if case == "almost":  # the changed tap is seen: 1e-6 of it reaches single pixels
        one = np.zeros((70, 90), np.float32)
        one[6, 5] = 1.0
        got = _blur(one, k)
        assert got[0, 0] == np.float32(k[0, 0]) and got[1, 1] == np.float32(k[1, 1])


def test_non_finite_images(gpu):
    rng = np.random.default_rng(4)
    img = rng.uniform(size=(40, 60)).astype(np.float32)
    img[5, 7], img[30, 40] = np.inf, np.nan
    k = np.outer(rng.uniform(0.5, 1.5, 6), rng.uniform(0.5, 1.5, 9))
    np.testing.assert_allclose(_blur(img, k), so.convolve_same(img, k), rtol=2 ** -23, atol=0)
