"""The batch tuner's own candidates: no two of them run the same kernels (they
would differ in the stack depth alone, which has no effect), and a cache written
with three numbers a candidate is still read."""
import json

import torch

import cubql_amd
from cubql_amd import autotune


def test_candidates_differ_in_what_has_an_effect():
    seen = [c[:2] for c in autotune.DEFAULT_CANDIDATES]
    assert len(seen) == len(set(seen))
    for c in autotune.DEFAULT_CANDIDATES:
        assert cubql_amd.BatchParams(*c).as_tuple() == (*c, 0)


def test_cached_choice(tmp_path, monkeypatch):
    monkeypatch.setattr(autotune, "_cache", {})
    monkeypatch.setattr(autotune, "_signature", lambda *a: "k")
    path = tmp_path / "tune.json"
    path.write_text(json.dumps({"k": {"best": [4, 128, 16], "times": {"(4, 128, 16)": 1.0}}}))
    off = torch.zeros(2, dtype=torch.int32)
    best, times = autotune.tune_batch(torch.zeros(0, 3), off, torch.zeros(0, 3), off, cache_path=str(path))
    assert best.as_tuple() == (4, 128, 16, 0) and times == {"(4, 128, 16)": 1.0}
