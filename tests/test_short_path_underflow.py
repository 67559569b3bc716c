"""A step time that underflows to zero ties with a time of zero: the full rule
then steps along y.  The short path (fast_group), which compares products, must
hand such a step back.  The field leads a line there in four steps: a fraction
of 2^-(3/2 top) beside a numerator of exactly zero, divided by the largest
velocity that the short path takes.  Compared bit for bit with the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from oracle_check import oracle_convolve
from rlic_amd import _core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pair_max", ["0", str(1 << 30)])
@pytest.mark.parametrize("klen", [17, 65])
# the exponents of the largest and smallest velocities, and of the fraction that
# the second step leaves
@pytest.mark.parametrize("dtype, top, frac", [(np.float32, 36, 50), (np.float64, 300, 290),
                                              (np.float64, 150, 290)])
def test_underflowing_step_time(monkeypatch, dtype, top, frac, klen, pair_max):
    two = dtype(2.0)
    rng = np.random.default_rng(klen)
    u = np.full((48, 48), 1.0, dtype)
    v = np.full((48, 48), 0.25, dtype)
    for i, j in ((5, 7), (20, 30), (33, 12), (40, 41)):  # the lines' start pixels
        u[i, j], v[i, j] = 1, two ** -top                          # x step to fx = 0
        u[i, j + 1], v[i, j + 1] = two ** (11 - frac), 1024        # y step: fx = 2^-frac, fy = 0
        u[i + 1, j + 1], v[i + 1, j + 1] = -(two ** top), two ** -top  # back in x: fx = 1, fy tiny
        u[i + 1, j], v[i + 1, j] = two ** top, -(two ** top)       # times 0 and, underflown, 0
    tex = rng.random((48, 48)).astype(dtype)
    kernel = rng.random(klen).astype(dtype)
    fn = _core.convolve_f32 if dtype == np.float32 else _core.convolve_f64
    monkeypatch.setenv("RLIC_TRACE_PAIR_MAX", pair_max)
    for iters in (1, 2):
        want = oracle_convolve(tex, u, v, kernel=kernel, uv_mode="velocity", iterations=iters,
                               boundaries={"x": "closed", "y": "closed"})
        got = fn(tex, (u, v, "velocity"), kernel, (("closed",) * 2,) * 2, iters)
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), int((got != want).sum())
