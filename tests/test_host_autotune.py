"""What the autotuner times and keeps, without a device: the sub-planes in
registers are among its candidates, at each split's own columns too, and the
library's own shape stays unless another is faster by more than runs differ."""
from __future__ import annotations

import pytest

import dfp
from dfp import autotune

OWN = (4, 0, 0, 0)


class _Array:
    def __init__(self, shape, zero=False):
        pass

    def download(self):
        return None

    def upload(self, a):
        pass


def _tune(monkeypatch, time_of):
    timed = []

    class _Plan:
        def __init__(self, g, device=0, precision=0, tuning=None):
            self.tuning = OWN if tuning is None else tuple(16 if i == 2 and tuning[3] == 1 and not v else v
                                                           for i, v in enumerate(tuning))

        def synth(self, *a, **k):
            pass

        def close(self):
            pass

    def time_plan(plan, fields, reps=10, warmup=3):
        timed.append(plan.tuning)
        return time_of(plan.tuning)

    monkeypatch.setattr(autotune, "Plan", _Plan)
    monkeypatch.setattr(autotune, "DeviceArray", _Array)
    monkeypatch.setattr(autotune, "time_plan", time_plan)
    return autotune.tune_plan(dfp.channel_grid(64, 32, 96, 1.5)), timed


def test_register_planes_are_candidates(monkeypatch):
    r, timed = _tune(monkeypatch, lambda t: 50.0 if t[2:] == (0, 0) and t[:2] == (8, 4) else 100.0)
    assert r["tuning"] == [8, 4, 0, 0] and r["us"] == 50.0 and r["default_us"] == 100.0
    for R in (1, 2, 3, 4, 6, 8, 12, 16):
        assert (R, 0, 0, 0) in timed
    assert any(t[3] == 2 for t in timed) and any(t[3] == 1 for t in timed)


@pytest.mark.parametrize("share,kept", [(0.99, True), (0.95, False)])
def test_the_librarys_shape_stays_within_the_noise(monkeypatch, share, kept):
    r, _ = _tune(monkeypatch, lambda t: 100.0 * share if t == (6, 8, 0, 2) else 100.0)
    assert r["tuning"] == (list(OWN) if kept else [6, 8, 0, 2])


def test_a_lucky_run_does_not_replace_the_librarys_shape(monkeypatch):
    runs = iter([30.0])
    r, _ = _tune(monkeypatch, lambda t: next(runs, 100.0) if t == (6, 8, 0, 2) else 100.0)
    assert r["tuning"] == list(OWN) and r["us"] == 100.0
