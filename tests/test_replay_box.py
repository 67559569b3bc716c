"""The replay from boxes cut to the lines (csrc/lic_replay_box.hip).

Every pass gathers the values that the tracing pass gathered, in the same
order, so the results are required bit for bit: against the oracle on small
fields, and against the L2-gather replay on a field where some tiles' boxes
do not fit the LDS.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import cpu
from rlic_amd import _core

pytestmark = pytest.mark.gpu


def _native(dtype):
    return _core.convolve_f32 if dtype == np.float32 else _core.convolve_f64


# partial and single tiles, rows of whole and of broken 16-byte quads, images
# smaller than a box (wrapped more than once)
SHAPES = [(1, 1), (3, 70), (32, 32), (37, 53), (64, 66), (100, 36)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("klen", [1, 2, 3, 17, 64, 65, 66, 131])
def test_against_oracle(dtype, shape, klen, monkeypatch):
    monkeypatch.setenv("RLIC_REPLAY_BOX", "2")
    rng = np.random.default_rng(klen + 1000 * shape[1])
    tex = rng.random(shape).astype(dtype)
    k = rng.random(klen).astype(dtype)
    for kind in ("random", "smooth", "holes"):
        u = (rng.random(shape) - 0.5).astype(dtype)
        v = (rng.random(shape) - 0.5).astype(dtype)
        if kind == "smooth":  # lines as long as the kernel
            u, v = (u * 0.2 + 1).astype(dtype), (v * 0.2 + 0.4).astype(dtype)
        elif kind == "holes":
            u[rng.random(shape) < 0.02] = np.nan
            v[rng.random(shape) < 0.02] = 0
        for mode, bx, by, iterations in (("velocity", "periodic", "periodic", 3),
                                         ("polarization", "closed", "periodic", 2),
                                         ("velocity", "closed", "closed", 4)):
            b = ((bx, bx), (by, by))
            exp = cpu.convolve(tex, u, v, kernel=k, uv_mode=mode,
                               boundaries={"x": bx, "y": by}, iterations=iterations, profile=1)
            got = _native(dtype)(tex, (u, v, mode), k, b, iterations, profile=1)
            assert np.array_equal(got, exp, equal_nan=True), (kind, mode, bx, by, iterations)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("klen", [129, 401])
@pytest.mark.parametrize("nx", [320, 301])
def test_boxes_that_do_not_fit(dtype, klen, nx, monkeypatch):
    """Saddles part the lines of a tile: one direction at a time, or the image."""
    ny = 288
    i, j = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    u = np.sin(i / 23.0).astype(dtype) + dtype(0.1)
    v = np.sin(j / 29.0).astype(dtype)
    rng = np.random.default_rng(klen)
    tex = rng.random((ny, nx)).astype(dtype)
    k = rng.random(klen).astype(dtype)
    b = (("periodic", "periodic"), ("closed", "closed"))
    monkeypatch.setenv("RLIC_REPLAY_BOX", "0")
    exp = _native(dtype)(tex, (u, v, "velocity"), k, b, 4)
    monkeypatch.setenv("RLIC_REPLAY_BOX", "2")
    got = _native(dtype)(tex, (u, v, "velocity"), k, b, 4)
    assert np.array_equal(got, exp)
