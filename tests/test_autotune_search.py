"""The autotuner's search on given timings (no GPU): a candidate replaces the
class's plan only if it is faster by more than the runs of either differ."""
import itertools
import json

import numpy as np
import pytest

from hyperflow_amd import autotune
from hyperflow_amd import case as C

CASE = C.quad_case(64, 64, 1, scheme="MUSCLHancock", limiter="VanLeer", cfl=0.5)


def search(tmp_path, monkeypatch, ms, cached=None):
    """tune() where plan (tile, tail, fix) takes ms(tile, tail, fix) plus 0, 1 % and 0.5 % in turn."""
    cache = tmp_path / "tuning.json"
    cls = autotune.problem_class(CASE, "fp32", "uniform")
    if cached:
        cache.write_text(json.dumps({autotune.class_key(cls): dict(zip(autotune.PARAMS, cached), ms_per_step=9.0,
                                                                   spread=0.0, **{"class": cls})}))
    monkeypatch.setattr(autotune, "CACHE", str(cache))
    noise = itertools.cycle((0.0, 0.01, 0.005))

    def run(cases, fields, precision, dt_mode, plan, steps, warmup, graph):
        return ms(*(plan[p] for p in autotune.PARAMS)) * (1.0 + next(noise)), "digest"

    monkeypatch.setattr(autotune, "_run", run)
    r = autotune.tune([CASE], [np.zeros(4)], precision="fp32", dt_mode="uniform", rows=(24, 8, 16), tails=(4, 8))
    assert autotune.cached_params(CASE, "fp32", "uniform") == {p: r[p] for p in autotune.PARAMS}
    return tuple(r[p] for p in autotune.PARAMS)


@pytest.mark.parametrize("cached", [None, (24, 8, 0)])
def test_equal_candidates_leave_the_plan(tmp_path, monkeypatch, cached):
    """All plans take the same time but for less than the runs differ."""
    best = search(tmp_path, monkeypatch, lambda tile, tail, fix: 1.0 - 0.004 * (tile == 8), cached)
    assert best == (cached or (24, 0, 0))


@pytest.mark.parametrize("cached", [None, (24, 8, 0)])
def test_faster_candidates_replace_it(tmp_path, monkeypatch, cached):
    best = search(tmp_path, monkeypatch, lambda tile, tail, fix: 1.0 - 0.1 * (tile == 16) - 0.05 * (tail == 4), cached)
    assert best == (16, 4, 0)
