"""The trace's full rule (full_group) and when it takes over: fields of ties,
zero components, lines that end or stay, tiny fractions and velocities at the
ends of the short path's range and beyond give the oracle's bits, whole and
partial groups, with and without the move record, both traces, all four
arithmetic profiles."""

from __future__ import annotations

import numpy as np
import pytest

from oracle_check import oracle_convolve, same_bits
from rlic_amd import _core

pytestmark = pytest.mark.gpu

PROFILES = {0: "none", 1: "fma", 2: "branchless", 3: "fma+branchless"}


def _field(kind, shape, dtype, rng):
    sign = lambda: rng.choice([-1.0, 1.0], shape)  # noqa: E731
    low, high = (-60, 40) if dtype == np.float32 else (-300, 150)
    if kind == "whole":  # ties, zeros of either sign, some ends
        u, v = (rng.integers(-2, 3, shape) * sign() for _ in range(2))
        u[rng.random(shape) < 0.005] = np.nan
    elif kind == "speckle":
        u, v = (rng.uniform(0.2, 1.5, shape) * sign() for _ in range(2))
        pick = rng.random(shape)
        u[pick < 0.02] = np.nan
        u[pick > 0.97], v[pick > 0.97] = 0.0, -0.0
    elif kind == "level":  # along x, sometimes just after a step along y
        u, v = rng.uniform(0.2, 1.5, shape) * sign(), 0.0 * sign()
        turn = rng.random(shape) < 0.3
        u[turn], v[turn] = 0.0, sign()[turn]
    elif kind == "ends":
        u, v = (np.exp2(rng.uniform(low, high, shape)) * sign() for _ in range(2))
        u[0, 0], v[0, 0] = 2.0 ** low, 2.0 ** high
    elif kind == "beyond":
        u, v = (np.exp2(rng.uniform(-20, 20, shape)) * sign() for _ in range(2))
        u[-1, -1] = 2.0 ** (low - 1)
        v[0, -1] = np.inf
    else:  # "tiny": steps that move the other axis by next to nothing
        mags = np.exp2(np.array([0.0, high - 1, low + 1]))
        u, v = (rng.choice(mags, shape, p=[0.4, 0.3, 0.3]) * sign() for _ in range(2))
    return u.astype(dtype), v.astype(dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["whole", "speckle", "level", "ends", "beyond", "tiny"])
def test_matches_the_oracle(monkeypatch, dtype, kind):
    rng = np.random.default_rng(len(kind) + 7 * ord(kind[0]))
    fn = _core.convolve_f32 if dtype == np.float32 else _core.convolve_f64
    cases = [((61, 83), 129, 2), ((61, 83), 42, 1), ((40, 37), 18, 3), ((1, 90), 33, 2),
             ((75, 1), 65, 2), ((2, 64), 81, 1), ((64, 2), 25, 2), ((3, 3), 129, 2)]
    for k, (shape, klen, iters) in enumerate(cases):
        u, v = _field(kind, shape, dtype, rng)
        tex, kernel = rng.random(shape).astype(dtype), rng.random(klen).astype(dtype)
        bounds = [("periodic", "closed"), ("closed", "periodic"), ("closed", "closed"),
                  ("periodic", "periodic")][k % 4]
        for mode in ("velocity", "polarization"):
            if kind == "beyond" and mode == "polarization":
                continue  # inf - inf: NaN signs are not defined
            for profile in (3,) if k > 1 else (3, 2, 1, 0):
                with np.errstate(all="ignore"):
                    want = oracle_convolve(tex, u, v, kernel=kernel, uv_mode=mode,
                                           iterations=iters, profile=PROFILES[profile],
                                           boundaries={"x": bounds[0], "y": bounds[1]})
                for pair_max in ("0", str(1 << 30)):
                    monkeypatch.setenv("RLIC_TRACE_PAIR_MAX", pair_max)
                    got = fn(tex, (u, v, mode), kernel, tuple((b, b) for b in bounds), iters,
                             profile=profile)
                    assert same_bits(got, want), (shape, klen, iters, mode, profile, pair_max)

