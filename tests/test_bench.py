"""The benchmark's timers: Python's collector does not run inside them."""

from __future__ import annotations

import gc

import pytest

import bench


def test_no_collection_while_a_timer_runs():
    runs = []

    def started(phase, info):
        if phase == "start":
            runs.append(info["generation"])

    def fill():
        assert not gc.isenabled()
        runs.clear()  # the collection before the timer
        keep = [[] for _ in range(200_000)]  # far past every generation's count
        assert runs == []
        return len(keep)

    gc.callbacks.append(started)
    try:
        assert bench.without_collection(fill)() == 200_000
        assert gc.isenabled()
        with pytest.raises(ZeroDivisionError):
            bench.without_collection(lambda: 1 // 0)()
        assert gc.isenabled()
    finally:
        gc.callbacks.remove(started)
    for timer in (bench.time_gpu, bench.time_gpu_spread):
        assert hasattr(timer, "__wrapped__")
