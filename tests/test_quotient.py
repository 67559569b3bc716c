"""The short path's quotient (quotient_rn) equals IEEE division over its range
of numerators and divisors, checked on the GPU against NumPy's division: random
operands, the ends of the range, quotients next to a rounding boundary and to a
power of two, exact ones, zero.  RLIC_EXHAUSTIVE=1 also tries every pair of
float mantissas (2^46)."""

from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from rlic_amd import _native

pytestmark = pytest.mark.gpu

# smallest numerator and divisor, largest divisor, as exponents
RANGE = {np.float32: (-60, -60, 40), np.float64: (-300, -300, 150)}


def _check(a: np.ndarray, b: np.ndarray) -> None:
    import torch

    dtype = a.dtype.type
    ta, tb = (torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0") for x in (a, b))
    tq = torch.empty_like(ta)
    lib = _native.load()
    fn = lib.rlic_quotient_check_f32 if dtype == np.float32 else lib.rlic_quotient_check_f64
    _native.raise_for_status(fn(ta.data_ptr(), tb.data_ptr(), tq.data_ptr(), ta.numel(), None))
    bits = np.uint32 if dtype == np.float32 else np.uint64
    got, want = tq.cpu().numpy().view(bits), (a / b).view(bits)
    bad = got != want
    assert not bad.any(), (int(bad.sum()), a[bad][:3], b[bad][:3])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_over_the_range(dtype):
    rng = np.random.default_rng(11)
    n_lo, d_lo, d_hi = RANGE[dtype]
    n = 1 << 22
    b = np.exp2(rng.uniform(d_lo, d_hi, n)).clip(2.0 ** d_lo, 2.0 ** d_hi).astype(dtype)
    tiny = np.exp2(rng.uniform(n_lo, 1, n)).clip(2.0 ** n_lo, 2).astype(dtype)
    usual = rng.uniform(2.0 ** -20, 1, n).astype(dtype)
    _check(tiny, b)
    _check(usual, b)
    _check(usual, rng.uniform(2.0 ** -10, 2, n).astype(dtype))
    ends_a = np.array([0.0, 2.0 ** n_lo, np.nextafter(dtype(2.0 ** n_lo), dtype(1)), 0.5, 1.0,
                       np.nextafter(dtype(1), dtype(0)), 1.5, 2.0], dtype)
    ends_b = np.array([2.0 ** d_lo, np.nextafter(dtype(2.0 ** d_lo), dtype(1)), 1.0, 3.0, 1 / 3,
                       np.nextafter(dtype(2.0 ** d_hi), dtype(0)), 2.0 ** d_hi], dtype)
    _check(np.repeat(ends_a, ends_b.size), np.tile(ends_b, ends_a.size))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_next_to_boundaries(dtype):
    rng = np.random.default_rng(12)
    eps = np.finfo(dtype).eps
    n = 1 << 21
    b = rng.uniform(1, 2, n).astype(dtype)
    # a next to b q: quotients on either side of q, exact ones among them
    for q in (rng.uniform(0.5, 1, n).astype(dtype), (1 - eps * rng.integers(0, 9, n)).astype(dtype),
              np.exp2(rng.integers(-20, 1, n)).astype(dtype)):
        a = (b * q).astype(dtype)
        for _ in range(3):
            _check(a, b)
            a = np.nextafter(a, dtype(0))
    # next to the middle between two quotients: b (q + half a unit), rounded
    q = (rng.integers(1 << 20, 1 << 21, n) / (1 << 21)).astype(dtype)
    half = (q.astype(np.longdouble) + np.longdouble(eps) / 4) * b.astype(np.longdouble)
    a = half.astype(dtype)
    for toward in (0, 4):
        _check(np.nextafter(a, dtype(toward)), b)
    _check(a, b)
    # divisors with mantissas of all ones or one
    for m in (dtype(2) - eps, dtype(1) + eps, dtype(1.5) - eps, dtype(1) + 3 * eps):
        _check(rng.uniform(0.25, 2, n).astype(dtype), np.full(n, m, dtype))


@pytest.mark.skipif(os.environ.get("RLIC_EXHAUSTIVE") != "1",
                    reason="14 s of GPU: RLIC_EXHAUSTIVE=1")
def test_every_pair_of_float_mantissas():
    import torch

    wrong = torch.zeros(1, dtype=torch.int64, device="cuda:0")
    step = 1 << 17
    for first in range(0, 1 << 23, step):
        st = _native.load().rlic_quotient_sweep_f32(first, step, ctypes.c_void_p(wrong.data_ptr()),
                                                    None)
        _native.raise_for_status(st)
        if first % (1 << 20) == 0:
            print(f"numerators up to {first + step}: {int(wrong)} wrong", flush=True)
    assert int(wrong) == 0


def test_a_part_of_the_sweep():
    import torch

    wrong = torch.zeros(1, dtype=torch.int64, device="cuda:0")
    for first, count in ((0, 64), ((1 << 23) - 64, 64), (5592405, 32)):
        st = _native.load().rlic_quotient_sweep_f32(first, count,
                                                    ctypes.c_void_p(wrong.data_ptr()), None)
        _native.raise_for_status(st)
    assert int(wrong) == 0
