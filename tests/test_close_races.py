"""Which options the full-graph decision times again as calls back to back
(no GPU: the timer is replaced)."""

from __future__ import annotations

import pytest

from autosage_amd import _auto


@pytest.mark.parametrize("times, again", [
    ({"null": 0.080, '"colslice"': 0.086}, {"null", '"colslice"'}),
    ({"null": 0.080, '"colslice"': 0.086, "[64, 2, 31]": 0.2}, {"null", '"colslice"'}),
    ({"null": 0.080, '"colslice"': 0.2}, set()),   # no race
    ({"null": 1.0, '"colslice"': 1.1}, set()),     # long calls
    ({"null": 0.080}, set()),
])
def test_short_calls_in_a_close_race_are_timed_again(monkeypatch, times, again):
    ran = []
    monkeypatch.setattr(_auto, "_time_cuda", lambda f, **kw: (f(), {"best_ms": 0.8})[1])
    got = _auto._back_to_back(dict(times), lambda option: ran.append(option))
    assert len(ran) == _auto._BURST * len(again)
    assert got == {k: (0.8 / _auto._BURST if k in again else v) for k, v in times.items()}
