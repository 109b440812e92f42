"""What the benchmark times is a plain pass: nothing observes its launches."""

import torch

import bench
from flash_model_architectures_amd import _native


def test_timed_steps_are_plain(monkeypatch):
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *args: None)
    observed = []

    def step():
        observed.append(_native.timeline_active())

    _, summary, passes = bench._time_steps(step, 12)
    assert observed == [False] * 12 + [True] * passes and 0 < passes <= bench.OBSERVED_PASSES and summary == {}
    assert not _native.timeline_active()
    observed.clear()
    assert bench._time_steps(step, 3, observe=False)[1:] == ({}, 0)
    assert observed == [False] * 3
