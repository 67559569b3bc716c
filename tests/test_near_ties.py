"""Fields in which every step of every line is a near tie of the same size: the
two step times differ by k halves of a unit in the last place, on either side of
where the trace's short path starts to trust their order (near_tie), for whole
waves, so that none of their steps is done again for another lane's sake.  Both
traces, with and without the move record, bit for bit against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from oracle_check import oracle_convolve, same_bits
from rlic_amd import _core

pytestmark = pytest.mark.gpu

SHAPE, KLEN = (45, 70), 65
HALVES = (0, 1, 2, 3, 5, 6, 7, 8, 9, 10, 12, 15, 16, 17, 18, 20, 33, 63, 65, 130)


@pytest.mark.parametrize("pair", ["131072", "0"])
@pytest.mark.parametrize("mode", ["velocity", "polarization"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_near_ties_of_a_given_size(monkeypatch, dtype, mode, pair):
    monkeypatch.setenv("RLIC_TRACE_PAIR_MAX", pair)
    rng = np.random.default_rng(21)
    fn = _core.convolve_f32 if dtype == np.float32 else _core.convolve_f64
    tex, kernel = rng.random(SHAPE).astype(dtype), rng.random(KLEN).astype(dtype)
    half = np.finfo(dtype).eps / 2
    bounds = (("periodic", "periodic"), ("closed", "closed"))
    for n, k in enumerate(HALVES):
        for sign in (1, -1):
            # one size for the field, then one for each row
            c = rng.uniform(0.5, 2.0, (1, 1) if n % 2 else (SHAPE[0], 1)) * np.ones(SHAPE)
            u = c.astype(dtype)
            v = (u.astype(np.longdouble) * (1 + k * half) * sign).astype(dtype)
            for a, b in ((u, v), (v, u)):
                for iterations in (1, 2):
                    got = fn(tex, (a, b, mode), kernel, bounds, iterations)
                    want = oracle_convolve(tex, a, b, kernel=kernel, uv_mode=mode,
                                           boundaries={"x": "periodic", "y": "closed"},
                                           iterations=iterations)
                    assert same_bits(got, want), (k, sign, iterations)
