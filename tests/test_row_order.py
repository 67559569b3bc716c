"""Row order of the guarded cell array (cell_slot): row pairs, and plain rows
where only those fit the allocation-free entry point's scratch (an odd number
of rows leaves half a pair unused).  Both give the oracle's bits, on images of
odd and even sides down to one pixel."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle_check import oracle_convolve
from rlic_amd import _core, _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(1, 1), (1, 70), (2, 33), (3, 3), (64, 1), (65, 2), (31, 66)])
def test_sides(monkeypatch, dtype, shape):
    rng = np.random.default_rng(shape[0] * 100 + shape[1])
    tex, u, v = (rng.random(shape).astype(dtype) - dtype(0.5) * k for k in (0, 1, 1))
    kernel = rng.random(41).astype(dtype)
    fn = _core.convolve_f32 if dtype == np.float32 else _core.convolve_f64
    for bounds in (("periodic", "closed"), ("closed", "periodic")):
        want = oracle_convolve(tex, u, v, kernel=kernel, iterations=2,
                               boundaries={"x": bounds[0], "y": bounds[1]})
        for pair_max in ("0", str(1 << 30)):
            monkeypatch.setenv("RLIC_TRACE_PAIR_MAX", pair_max)
            got = fn(tex, (u, v, "velocity"), kernel, tuple((b, b) for b in bounds), 2)
            assert np.array_equal(got, want), (bounds, pair_max)


@pytest.mark.parametrize("iterations", [1, 2])
def test_plain_rows_where_pairs_do_not_fit(gpu_device, iterations):
    """5 rows of 700002 cells of 16 bytes (and the ping-pong buffer) fit the
    64 MiB; 6 rows do not."""
    import torch

    shape, klen = (3, 700000 if iterations == 2 else 830000), 17
    rng = np.random.default_rng(iterations)
    tex = rng.random(shape).astype(np.float32)
    u, v = ((rng.random(shape) - 0.5).astype(np.float32) for _ in range(2))
    kernel = rng.random(klen).astype(np.float32)
    t = [torch.from_numpy(a).to(gpu_device) for a in (tex, u, v, kernel)]
    out = torch.full_like(t[0], float("nan"))
    nx = shape[1]
    status = _native.load().rlic_convolve_noalloc_f32(
        t[0].data_ptr(), nx, 1, t[1].data_ptr(), nx, 1, t[2].data_ptr(), nx, 1, shape[0], nx,
        t[3].data_ptr(), klen, 0, 1, 1, 0, 0, iterations, out.data_ptr(), 3,
        ctypes.c_void_p(torch.cuda.current_stream(gpu_device).cuda_stream))
    assert status == 0, _native.last_error()
    want = oracle_convolve(tex, u, v, kernel=kernel, iterations=iterations,
                           boundaries={"x": "periodic", "y": "closed"})
    assert np.array_equal(out.cpu().numpy(), want)
