"""The batched launch gives the bits of single calls for every work-item
region side, with fewer items than waves (every item taken by a wave's
number) and with more (popped from the queue), and for batches whose fields
leave after different numbers of passes."""

from __future__ import annotations

import numpy as np
import pytest

import rlic_amd
from rlic_amd.batch import convolve_batch

pytestmark = pytest.mark.gpu


def _fields(dtype, shapes, device):
    import torch

    rng = np.random.default_rng(len(shapes))
    fields = []
    for k, (ny, nx) in enumerate(shapes):
        tex, u, v = (torch.from_numpy((rng.random((ny, nx)) - 0.5 * (j > 0)).astype(dtype)).to(device)
                     for j in range(3))
        kernel = torch.from_numpy(rng.random(9 + 8 * (k % 5)).astype(dtype)).to(device)
        fields.append(dict(texture=tex, u=u, v=v, kernel=kernel,
                           uv_mode=("velocity", "polarization")[k % 2],
                           boundaries={"x": ("closed", "periodic")[k % 2],
                                       "y": ("periodic", "closed")[k // 2 % 2]},
                           iterations=k % 4 + (k > 0)))
    return fields


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("side", ["", "8", "16", "32", "64"])
@pytest.mark.parametrize("shapes", [[(1, 1), (7, 9), (33, 64), (65, 20), (8, 8)],
                                    [(300 + k, 310 - 7 * k) for k in range(9)]])
def test_regions(monkeypatch, gpu_device, dtype, side, shapes):
    monkeypatch.setenv("RLIC_BATCH_REGION", side)
    fields = _fields(dtype, shapes, gpu_device)
    for k, (got, f) in enumerate(zip(convolve_batch(fields), fields)):
        args = (f.pop("texture"), f.pop("u"), f.pop("v"))
        want = rlic_amd.convolve(*args, **f)
        assert np.array_equal(got.cpu().numpy(), want.cpu().numpy()), (k, shapes[k])
