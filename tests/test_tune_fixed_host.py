"""A split rule stored as fixed (chosen from layers of mixed sizes, which the tuner does
not time) survives a re-tune; without the mark the tuner's own rule is stored."""
import json

import pytest

from test_tune_host import _fake_engine


@pytest.mark.parametrize("fixed", [False, True])
def test_fixed_split_rule_survives_a_retune(tmp_path, fixed):
    from mpsim_amd import tune

    def timer(eng, items, cfg, reps):  # two groups are the fastest, whatever the batch
        return {1: 1.0, 2: 0.5, 3: 0.7, 4: 0.8}[eng.split_ways]

    path = str(tmp_path / "tuned.json")
    rule = {"split_ways": 4, "split_rows": 257, "split_min": 1}
    with open(path, "w") as f:
        json.dump(dict(rule, split_fixed=1) if fixed else rule, f)
    out = tune.tune(_fake_engine(), chis=(8, 64), reps=1, path=path, conc_chis=(64,), layer=4, timer=timer)
    assert tune.tuned_engine(path) == ((4, 1, 257) if fixed else (2, 2, 128))
    assert bool(out.get("split_fixed")) == fixed
    assert {r["stage"] for r in out["measurements"]} >= {"split", "split_min"}  # measured either way


def test_stored_rule_is_marked():
    """The rule in the repository cannot come out of the tuner (its classes are
    2 chi rows, its batches two problems and more)."""
    from mpsim_amd import tune
    stored = tune._load(tune.TUNED)
    if stored.get("split_min") == 1 or stored.get("split_rows", 0) % 2:
        assert stored.get("split_fixed")


def test_pivot_stage_times_what_has_pivots(tmp_path):
    """The default method has no pivots up to 1024 rows (its options would be
    chosen by noise): the pivot stage asks for the one-sided rounds."""
    from mpsim_amd import tune
    seen = []

    def timer(eng, items, cfg, reps):
        if cfg.block:
            seen.append(cfg.method)
        return 1.0

    tune.tune(_fake_engine(), chis=(8, 64), reps=1, path=str(tmp_path / "t.json"), conc_chis=(), timer=timer)
    assert seen == [1] * 8
