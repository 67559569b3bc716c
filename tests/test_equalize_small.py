"""Equalization of small images, where one or a few blocks take part in every
launch, and of more bins than pixels or than a block's LDS holds: global, per
window and interpolated, against the oracle, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

import rlic_amd
from oracle import equalize as eq
from rlic_amd.equalize import (equalize_histogram_sliding_tile,
                               equalize_histogram_tile_interpolation)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nbins", [1, 3, 256, 16384, 16385, 70000])
@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (64, 33), (257, 250)])
def test_small_images(gpu_device, dtype, nbins, shape):
    import torch

    rng = np.random.default_rng(nbins + shape[1])
    img = rng.normal(size=shape).astype(dtype)
    if img.size > 1:
        img[rng.random(shape) < 0.05] = np.nan
        img[-1, 0] = np.inf
    for values in (img, np.full(shape, np.nan, dtype), np.full(shape, 2.5, dtype)):
        t = torch.from_numpy(values).to(gpu_device)
        for view, a in ((t, values), (t.T, values.T)):
            got = rlic_amd.equalize_histogram(view, nbins).cpu().numpy()
            assert np.array_equal(got, eq.equalize_histogram(a, nbins), equal_nan=True)
    if img.size <= 64 * 33 and nbins <= 256:
        t = torch.from_numpy(img).to(gpu_device)
        for ours, oracle in ((equalize_histogram_sliding_tile, eq.equalize_histogram_sliding_tile),
                             (equalize_histogram_tile_interpolation,
                              eq.equalize_histogram_tile_interpolation)):
            got = ours(t, nbins, (9, 7)).cpu().numpy()
            assert np.array_equal(got, oracle(img, nbins, (9, 7)), equal_nan=True)
