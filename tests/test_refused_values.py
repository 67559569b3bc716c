"""A convolve call whose values are refused (src/rlic/_lib.py:174, :194) does
not compute: no trace or replay runs on a large one, no replay plan is measured
and kept from it, and the next call gives the oracle's bits."""

from __future__ import annotations

import numpy as np
import pytest

import rlic_amd
from rlic_amd import _native

pytestmark = pytest.mark.gpu


def _inputs(ny, nx, klen, dtype):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(klen)
    draw = lambda *s: torch.rand(*s, generator=gen, device="cuda", dtype=dtype)  # noqa: E731
    return draw(ny, nx), draw(ny, nx) - 0.5, draw(ny, nx) - 0.5, draw(klen)


@pytest.mark.parametrize("bad", ["texture", "kernel", "both"])
@pytest.mark.parametrize("dtype, n, iters", [("float32", 2048, 4), ("float64", 2048, 2),
                                             ("float32", 4096, 1)])
def test_large_refused_call_runs_nothing(bad, dtype, n, iters):
    import torch

    tex, u, v, kernel = _inputs(n, n, 131, getattr(torch, dtype))  # at least 2^31 steps
    if bad != "kernel":
        tex[n // 2, 3] = -1
    if bad != "texture":
        kernel[7] = float("inf")
    _native.profiler_enable(True)
    try:
        _native.profiler_read()
        with pytest.raises(Exception) as err:
            rlic_amd.convolve(tex, u, v, kernel=kernel, iterations=iters)
        torch.cuda.synchronize()
        ran = _native.profiler_read()
    finally:
        _native.profiler_enable(False)
    assert {k for k in ran if "trace" in k or "replay" in k} == set()
    assert len(getattr(err.value, "exceptions", [err.value])) == (2 if bad == "both" else 1)


def test_no_plan_is_measured_on_refused_values(monkeypatch):
    import torch

    from oracle_check import oracle_convolve, same_bits

    monkeypatch.setenv("RLIC_AUTOTUNE", "1")
    _native.autotune_clear()
    tex, u, v, kernel = _inputs(520, 530, 33, torch.float32)
    kw = dict(kernel=kernel, boundaries="periodic", iterations=3)
    tex[5, 5] = -0.25
    with pytest.raises(ValueError, match="invalid texture"):
        rlic_amd.convolve(tex, u, v, **kw)
    assert _native.autotune_table() == []
    tex[5, 5] = 0.25
    got = rlic_amd.convolve(tex, u, v, **kw)
    assert len(_native.autotune_table()) == 1
    assert same_bits(got.cpu().numpy(), oracle_convolve(tex, u, v, **kw))
    _native.autotune_clear()
