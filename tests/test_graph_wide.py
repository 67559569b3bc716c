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


@pytest.mark.parametrize("dtype, tiny", [(np.float32, 1e-42), (np.float64, 1e-310)])
@pytest.mark.parametrize("iterations, replay, pair", [(1, "1", True), (1, "1", False),
                                                      (3, "1", False), (3, "0", True)])
def test_fields_of_any_range_in_turn(gpu_device, monkeypatch, dtype, tiny, iterations, replay, pair):
    """One graph, its inputs changed between fields within the short path's
    range and out of it, with eager calls of other sizes between the replays
    (they leave other values where the graph's call counts its replays)."""
    import torch

    monkeypatch.setenv("RLIC_REPLAY", replay)
    monkeypatch.setenv("RLIC_TRACE_PAIR_MAX", "131072" if pair else "0")
    lib = _native.load()
    fn = lib.rlic_convolve_noalloc_f32 if dtype is np.float32 else lib.rlic_convolve_noalloc_f64
    ny, nx, klen = 61, 83, 33
    rng = np.random.default_rng(11)
    fields = [rng.standard_normal((2, ny, nx)) for _ in range(3)]
    fields[1] *= tiny
    fields[2][:, 5, 7] = np.inf
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype)).to(gpu_device)  # noqa: E731
    tex, u, v, k = on(rng.random((ny, nx))), on(fields[0][0]), on(fields[0][1]), on(rng.random(klen))
    out = torch.empty_like(tex)
    other = [on(rng.random((70, 40))) for _ in range(4)]

    def call(t, a, b, dest):
        stream = torch.cuda.current_stream(gpu_device).cuda_stream
        h, w = t.shape
        st = fn(t.data_ptr(), w, 1, a.data_ptr(), w, 1, b.data_ptr(), w, 1, h, w, k.data_ptr(), klen,
                0, 1, 1, 0, 0, iterations, dest.data_ptr(), 3, ctypes.c_void_p(stream))
        assert st == 0, _native.last_error()

    side = torch.cuda.Stream(gpu_device)
    with torch.cuda.stream(side):
        call(tex, u, v, out)
    side.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=side):
        call(tex, u, v, out)
    if iterations == 1:  # packing and the trace, nothing else
        nodes = ctypes.c_size_t()
        assert lib.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None,
                                    ctypes.byref(nodes)) == 0
        assert nodes.value == 2
    graph.instantiate()
    bounds = {"x": "periodic", "y": "closed"}
    wants = []
    for f in fields:
        u.copy_(on(f[0]))
        v.copy_(on(f[1]))
        wants.append(oracle_convolve(tex, u, v, kernel=k, boundaries=bounds, iterations=iterations))
    for turn, which in enumerate((0, 1, 0, 0, 2, 1, 1, 0, 2, 0)):
        u.copy_(on(fields[which][0]))
        v.copy_(on(fields[which][1]))
        if turn % 3 == 2:
            call(other[2], other[0], other[1], other[3])
        graph.replay()
        torch.cuda.synchronize(gpu_device)
        assert same_bits(out.cpu().numpy(), wants[which]), (turn, which)
