"""The trace's short path (one division per step, the axis picked by a cross
product: fast_group) gives the bits of the full rule, i.e. of the oracle:
fields made of near and exact ties, of components at the ends of the range
it takes and beyond them, of fractions so small that it must step back, and
of lines that end or stay, with both traces, whole and partial chunks, with
and without the move record.  Results are compared bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from oracle_check import oracle_convolve
from rlic_amd import _core

pytestmark = pytest.mark.gpu

SHAPE = (61, 83)


def _field(kind, dtype, rng):
    one = rng.uniform(0.3, 1.5, SHAPE) * rng.choice([-1, 1], SHAPE)
    # ends of the accepted range: 2^-40..2^40 in float, 2^-300..2^300 in double
    top = 40 if dtype == np.float32 else 300
    if kind == "near_ties":  # |u| and |v| within a few units in the last place
        u = one.astype(dtype)
        off = rng.integers(-40, 41, SHAPE) * np.finfo(dtype).eps
        v = (u * (1 + off).astype(dtype) * rng.choice([-1, 1], SHAPE)).astype(dtype)
    elif kind == "ties":
        u = np.ones(SHAPE, dtype)
        v = np.ones(SHAPE, dtype)
    elif kind in ("range", "beyond"):
        u, v = (np.exp2(rng.uniform(-top, top, SHAPE)) * rng.choice([-1, 1], SHAPE)
                for _ in range(2))
        u, v = u.astype(dtype), v.astype(dtype)
        u[3, 5], v[3, 5] = dtype(2.0) ** top, -(dtype(2.0) ** -top)
        if kind == "beyond":
            u[7, 9], v[40, 11], u[20, 60] = dtype(2.0) ** -(top + 1), dtype(2.0) ** (top + 1), np.inf
    elif kind == "small_fractions":  # steps that move the other axis by 2^-(7/4 top)
        mags = np.exp2(np.array([0.0, 0.875 * top, -0.875 * top]))
        u, v = (rng.choice(mags, SHAPE) * rng.choice([-1, 1], SHAPE) for _ in range(2))
    else:  # lines that end (NaN), stay (zero vectors), move along one axis
        u, v = one.copy(), (one * rng.uniform(-1, 1, SHAPE))
        pick = rng.random(SHAPE)
        u[pick < 0.02], v[(pick > 0.01) & (pick < 0.03)] = np.nan, np.nan
        zero = (pick > 0.95) | (np.add.outer(np.arange(SHAPE[0]) // 8, np.arange(SHAPE[1]) // 8) % 7 == 0)
        u[zero], v[zero] = 0.0, -0.0
        u[(pick > 0.5) & (pick < 0.6)] = -0.0
    return u.astype(dtype), v.astype(dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["near_ties", "ties", "range", "beyond", "small_fractions", "stops"])
def test_short_path_matches(monkeypatch, dtype, kind):
    rng = np.random.default_rng(sum(map(ord, kind)))
    tex = rng.random(SHAPE).astype(dtype)
    u, v = _field(kind, dtype, rng)
    fn = _core.convolve_f32 if dtype == np.float32 else _core.convolve_f64
    modes = ("velocity",) if kind == "beyond" else ("velocity", "polarization")
    for mode in modes:
        for klen, iters, bounds in ((129, 2, ("periodic", "closed")), (41, 1, ("closed", "periodic")),
                                    (17, 3, ("periodic", "periodic")), (64, 1, ("closed", "closed"))):
            kernel = rng.random(klen).astype(dtype)
            with np.errstate(all="ignore"):
                want = oracle_convolve(tex, u, v, kernel=kernel, uv_mode=mode, iterations=iters,
                                       boundaries={"x": bounds[0], "y": bounds[1]})
            for pair_max in ("0", str(1 << 30)):
                monkeypatch.setenv("RLIC_TRACE_PAIR_MAX", pair_max)
                got = fn(tex, (u, v, mode), kernel, tuple((b, b) for b in bounds), iters)
                assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), \
                    (mode, klen, iters, bounds, pair_max, int((got != want).sum()))
