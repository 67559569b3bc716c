"""The replay autotuner keeps plans by whether boxes cut to the lines were among
the candidates, which depends on the number of passes: a call of few passes does
not decide for one of many, whatever their order, and tables written without
that mark load as before."""

from __future__ import annotations

import numpy as np
import pytest

import rlic_amd
from rlic_amd import _native


@pytest.mark.gpu
def test_few_passes_do_not_decide_for_many(monkeypatch, tmp_path):
    import torch

    monkeypatch.setenv("RLIC_REPLAY_LDS", "1")
    monkeypatch.setenv("RLIC_AUTOTUNE", "1")
    cache = tmp_path / "plans.txt"
    monkeypatch.setenv("RLIC_AUTOTUNE_CACHE", str(cache))
    _native.autotune_clear()
    rng = np.random.default_rng(5)
    ny, nx, klen = 1024, 1024, 129  # half length 64: boxes from 4 replays on
    t = lambda a: torch.from_numpy(a.astype(np.float32)).to("cuda:0")  # noqa: E731
    y, x = np.mgrid[:ny, :nx] * (2 * np.pi / ny)
    tex, u, v = t(rng.random((ny, nx))), t(np.cos(3 * x) + 0.2), t(np.sin(2 * y) + 0.7)
    kw = dict(kernel=t(rng.random(klen)), boundaries="periodic")
    table = lambda: {e["boxes"]: e for e in _native.autotune_table()}  # noqa: E731
    rlic_amd.convolve(tex, u, v, iterations=3, **kw)
    assert set(table()) == {False}
    _native.profiler_enable(True)
    try:
        out = rlic_amd.convolve(tex, u, v, iterations=12, **kw)
        assert set(table()) == {False, True}  # measured again, with boxes
        few = dict(table()[False])
        rlic_amd.convolve(tex, u, v, iterations=3, **kw)
        rlic_amd.convolve(tex, u, v, iterations=12, **kw)
    finally:
        _native.profiler_enable(False)
        _native.profiler_read()
    assert table()[False] == few
    lines = cache.read_text().splitlines()
    assert [ln.split()[-2:] for ln in lines] == [["boxes", "0"], ["boxes", "1"]]
    # a table that only knows calls without boxes does not keep them out
    _native.autotune_clear()
    old = tmp_path / "old.txt"
    old.write_text(f"rlic-replay-plan 4 {ny} {nx} {klen} 3 0 0 0 4 3 0.001\n")
    assert _native.autotune_load(old) == 1
    again = rlic_amd.convolve(tex, u, v, iterations=12, **kw)
    assert set(table()) == {False, True}
    assert torch.equal(out, again)
    # the box plan, loaded
    _native.autotune_clear()
    old.write_text(f"rlic-replay-plan 4 {ny} {nx} {klen} 3 2 32 32 0 0 0.001\n")
    assert _native.autotune_load(old) == 1
    assert torch.equal(out, rlic_amd.convolve(tex, u, v, iterations=12, **kw))
    assert set(table()) == {True}
    _native.autotune_clear()


def test_tables_with_and_without_the_mark(tmp_path):
    path = tmp_path / "plans.txt"
    path.write_text("rlic-replay-plan 4 512 600 129 3 1 64 64 0 0 0.5\n"
                    "rlic-replay-plan 4 512 600 129 3 2 32 32 0 0 0.25\n"
                    "rlic-replay-plan 4 512 700 129 3 0 0 0 16 3 0.25 boxes 1\n"
                    "rlic-replay-plan 4 512 700 129 3 2 64 64 64 0 0.75 boxes 0")
    _native.autotune_clear()
    assert _native.autotune_load(path) == 4
    got = {(e["nx"], e["boxes"]): e["pass_ms"] for e in _native.autotune_table()}
    assert got == {(600, False): 0.5, (600, True): 0.25, (700, True): 0.25, (700, False): 0.75}
    _native.autotune_clear()


@pytest.mark.gpu
def test_box_replays_are_told_apart(monkeypatch, tmp_path):
    import torch

    monkeypatch.setenv("RLIC_REPLAY_LDS", "1")
    monkeypatch.setenv("RLIC_REPLAY_BOX", "2")
    monkeypatch.setenv("RLIC_AUTOTUNE", "0")
    rng = np.random.default_rng(8)
    t = lambda *s: torch.from_numpy(rng.random(s).astype(np.float32)).to("cuda:0")  # noqa: E731
    _native.profiler_enable(True)
    _native.profiler_read()
    try:
        rlic_amd.convolve(t(90, 70), t(90, 70), t(90, 70), kernel=t(33), iterations=4)
        ran = _native.profiler_read()
    finally:
        _native.profiler_enable(False)
    assert {k for k in ran if "replay" in k} == {"lic_replay_lds"}
    replays = ran["lic_replay_lds"]
    assert replays["count"] == replays["box_count"] == 3
    assert replays["box_ms"] == replays["total_ms"] > 0


def test_the_box_plan_has_a_name(tmp_path):
    path = tmp_path / "plans.txt"
    path.write_text("rlic-replay-plan 4 512 600 129 3 2 32 32 0 0 0.25\n")
    _native.autotune_clear()
    assert _native.autotune_load(path) == 1
    assert [e["replay"] for e in _native.autotune_table()] == ["lds_box"]
    _native.autotune_clear()
