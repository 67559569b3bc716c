"""A captured allocation-free call replayed on a field with components beyond
the short path's range, and then on others: the replays that follow are as fast
as those before (the mark of the wide field does not stay), and every one gives
the oracle's bits."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle_check import oracle_convolve, same_bits
from rlic_amd import _native

pytestmark = pytest.mark.gpu


def test_a_wide_field_does_not_slow_later_replays(gpu_device):
    import torch

    lib = _native.load()
    n, klen = 1024, 129
    rng = np.random.default_rng(4)
    y, x = np.mgrid[:n, :n] * (2 * np.pi / n)
    u = np.cos(3 * x + y) + 0.4 * np.sin(5 * y)
    v = np.sin(2 * x - 3 * y) + 0.3 * np.cos(4 * x + 1)
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(gpu_device)  # noqa: E731
    tex, tu, tv, k = on(rng.random((n, n))), on(u), on(v), on(rng.random(klen))
    out = torch.empty_like(tex)

    def call():
        stream = torch.cuda.current_stream(gpu_device).cuda_stream
        st = lib.rlic_convolve_noalloc_f32(
            tex.data_ptr(), n, 1, tu.data_ptr(), n, 1, tv.data_ptr(), n, 1, n, n, k.data_ptr(), klen,
            0, 1, 1, 0, 0, 1, out.data_ptr(), 3, ctypes.c_void_p(stream))
        assert st == 0, _native.last_error()

    side = torch.cuda.Stream(gpu_device)
    with torch.cuda.stream(side):
        call()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call()

    def replay():
        """Best time of a few replays, after one; the output is checked."""
        graph.replay()
        times = []
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(4):
                graph.replay()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        rows = (500, 503)
        want = oracle_convolve(tex, tu, tv, kernel=k, boundaries={"x": "periodic", "y": "closed"},
                               rows=rows)
        assert same_bits(out[rows[0]:rows[1]].cpu().numpy(), want[rows[0]:rows[1]])
        return min(times)

    before = replay()
    tu[7, 9] = 1e-42
    replay()
    tu[7, 9] = 0.5
    after = replay()
    # the full rule takes 1.3 times as long as the short path
    assert after < 1.15 * before, (before, after)
