"""The element checks made while the convolution runs (rlic_convolve_checked_*).

Values that are refused are refused as before, with the same errors, and
results are those of the check and the convolution called one after the other.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import rlic_amd
from rlic_amd import _core

pytestmark = pytest.mark.gpu

NEGATIVE = "Found invalid texture element"
NON_FINITE = "Found non-finite value"


def _field(shape, dtype, klen, seed=0):
    g = torch.Generator().manual_seed(seed)
    tex, u, v = (torch.rand(shape, generator=g, dtype=dtype) for _ in range(3))
    return tex.cuda(), (u - 0.5).cuda(), (v - 0.5).cuda(), torch.rand(klen, dtype=dtype).cuda()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(1, 1), (63, 65), (700, 513)])
@pytest.mark.parametrize("iterations", [1, 3])
def test_values_refused(dtype, shape, iterations):
    tex, u, v, k = _field(shape, dtype, 17)
    call = dict(kernel=k, iterations=iterations)
    native = _core.convolve_f32 if dtype == torch.float32 else _core.convolve_f64
    closed = (("closed", "closed"), ("closed", "closed"))
    want = native(tex, (u, v, "velocity"), k, closed, iterations)
    for i, j in ((0, 0), (shape[0] - 1, shape[1] - 1), (shape[0] // 2, 0)):
        bad = tex.clone()
        bad[i, j] = -1e-30
        with pytest.raises(ValueError, match=NEGATIVE):
            rlic_amd.convolve(bad, u, v, **call)
        bad[i, j] = float("nan")  # not below 0
        rlic_amd.convolve(bad, u, v, **call)
        bad[i, j] = -0.0
        rlic_amd.convolve(bad, u, v, **call)
    for t, value in ((0, float("inf")), (8, float("nan")), (16, float("-inf"))):
        bad_k = k.clone()
        bad_k[t] = value
        with pytest.raises(ValueError, match=NON_FINITE):
            rlic_amd.convolve(tex, u, v, kernel=bad_k, iterations=iterations)
        bad = tex - 2
        with pytest.raises(Exception, match="Invalid inputs were received") as info:
            rlic_amd.convolve(bad, u, v, kernel=bad_k, iterations=iterations)
        assert [str(e)[:20] for e in info.value.exceptions] == [NEGATIVE[:20], NON_FINITE[:20]]
    # the flags of a refused call are not seen by the next one
    assert torch.equal(rlic_amd.convolve(tex, u, v, **call), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_strided_inputs_and_streams(dtype):
    tex, u, v, k = _field((130, 190), dtype, 34, seed=1)
    views = [t.t()[::2, 3:].flip(0).contiguous() if n == 0 else t.t()[::2, 3:].flip(0)
             for n, t in enumerate((tex, u, v))]
    want = rlic_amd.convolve(*(w.cpu().numpy() for w in views), kernel=k.cpu().numpy(),
                             iterations=2)
    texture = tex.t()[::2, 3:].flip(0)
    texture = torch.empty(95, 254, dtype=dtype, device="cuda")[:, ::2].copy_(texture)
    got = []
    for s in (torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.current_stream()):
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            got.append(rlic_amd.convolve(texture, views[1], views[2], kernel=k[:], iterations=2))
    torch.cuda.synchronize()
    for g in got:
        assert np.array_equal(g.cpu().numpy(), want)
