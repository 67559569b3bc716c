"""Kernels about the length of the trace's first whole group of 8 steps, below
which no short path is prepared, by single calls with both traces and in a
batch, with and without the move record, bit for bit against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from oracle_check import oracle_convolve, same_bits
from rlic_amd import _core
from rlic_amd.batch import Field, convolve_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["velocity", "polarization"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_short_kernels(monkeypatch, gpu_device, dtype, mode):
    import torch

    rng = np.random.default_rng(3)
    fn = _core.convolve_f32 if dtype == np.float32 else _core.convolve_f64
    ny, nx = 37, 53
    tex = rng.random((ny, nx)).astype(dtype)
    u, v = (rng.standard_normal((ny, nx)).astype(dtype) for _ in range(2))
    u[5, 7], v[20, 30], u[30, 11] = np.nan, 0.0, 0.0
    v[30, 11] = 0.0
    bounds = {"x": "periodic", "y": "closed"}
    fields, wants = [], []
    on = lambda a: torch.from_numpy(a).to(gpu_device)  # noqa: E731
    for klen in (1, 2, 3, 8, 9, 14, 15, 16, 17, 18, 19):
        kernel = rng.random(klen).astype(dtype)
        for iterations in (1, 2):
            want = oracle_convolve(tex, u, v, kernel=kernel, uv_mode=mode, boundaries=bounds,
                                   iterations=iterations)
            for pair in ("0", "131072"):
                monkeypatch.setenv("RLIC_TRACE_PAIR_MAX", pair)
                got = fn(tex, (u, v, mode), kernel, (("periodic",) * 2, ("closed",) * 2), iterations)
                assert same_bits(got, want), (klen, iterations, pair)
            fields.append(Field(on(tex), on(u), on(v), on(kernel), uv_mode=mode, boundaries=bounds,
                                iterations=iterations))
            wants.append(want)
    for f, got, want in zip(fields, convolve_batch(fields), wants):
        assert same_bits(got.cpu().numpy(), want), (f.kernel.numel(), f.iterations)
