"""Which options the full-graph decision times again as calls back to back, and
that one basis decides, is recorded and meets the baseline (no GPU: the timer is
replaced)."""

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


@pytest.mark.parametrize("alone, back_to_back, choice, candidate", [
    # the burst's winner, which alone is behind the baseline
    ({None: 0.080, "colslice": 0.086, "base": 0.083}, {None: 0.073, "colslice": 0.063, "base": 0.081}, "autosage", "colslice"),
    # behind the baseline only as calls back to back
    ({None: 0.080, "colslice": 0.086, "base": 0.090}, {None: 0.073, "colslice": 0.075, "base": 0.070}, "baseline", None),
    # the exact one within the margin
    ({None: 0.080, "colslice": 0.078, "base": 0.9}, {None: 0.072, "colslice": 0.070, "base": 0.9}, "autosage", None),
    # long calls: alone, all of them
    ({None: 2.0, "colslice": 1.5, "base": 1.4}, {}, "baseline", None),
    ({None: 2.0, "colslice": 1.5, "base": 1.6}, {}, "autosage", "colslice"),
])
def test_one_basis_decides_and_is_recorded(monkeypatch, alone, back_to_back, choice, candidate):
    ran = []

    def timer(f, **kw):
        del ran[:]
        f()
        assert len(set(ran)) == 1
        return {"best_ms": alone[ran[0]] if len(ran) == 1 else len(ran) * back_to_back[ran[0]]}

    monkeypatch.setattr(_auto, "_time_cuda", timer)
    result = {}
    _auto._decide_on_full_graph(result, [None, "colslice"], ran.append, lambda: ran.append("base"), inexact=("colslice",))
    assert (result["choice"], result["candidate"]) == (choice, candidate)
    record = result["full_graph"]
    basis = back_to_back or alone
    assert {c["candidate"]: c["best_ms"] for c in record["candidates"]} == {k: basis[k] for k in (None, "colslice")}
    assert record["baseline_ms"] == basis["base"] and record["back_to_back"] == bool(back_to_back)
    assert (result["choice"] == "autosage") == (record["autosage_ms"] <= record["baseline_ms"])
    assert record["autosage_ms"] in (basis[None], basis["colslice"])
