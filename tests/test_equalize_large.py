"""Global equalization of images large enough for every launch shape of its
kernels (partial ranges of the most blocks, eight loads in flight and their
remainder, the histogram's and the value table's bin limits), contiguous and
strided, against the oracle, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

import rlic_amd
from oracle import equalize as eq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nbins", [256, 2048, 2049])
@pytest.mark.parametrize("shape", [(2051, 2113), (700, 3001), (1, 5000), (4099, 1)])
def test_shapes(gpu_device, dtype, nbins, shape):
    import torch

    rng = np.random.default_rng(nbins + shape[0])
    img = rng.normal(size=shape).astype(dtype)
    img[rng.random(shape) < 0.001] = np.nan
    want = eq.equalize_histogram(img, nbins)
    flat = torch.from_numpy(img).to(gpu_device)
    wide = torch.full((shape[0], shape[1] + 3), 7.0, dtype=flat.dtype, device=gpu_device)
    wide[:, 1:-2] = flat
    for t in (flat, wide[:, 1:-2]):
        got = rlic_amd.equalize_histogram(t, nbins)
        assert np.array_equal(got.cpu().numpy(), want, equal_nan=True)
