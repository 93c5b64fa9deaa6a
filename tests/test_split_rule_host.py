"""Which rule decides whether a two-site call is split over streams: the stored one for
the direct solver, the stored one of the rounds for methods that iterate at every
size, and a rule that the caller sets for both."""
import json

import pytest

ROUNDS = (dict(method=1), dict(fp32=True), dict(fp32_sweeps=12), dict(block=8))


def _engine(tmp_path, stored):
    from mpsim_amd import tune
    from mpsim_amd.engine import Engine
    path = str(tmp_path / "tuned.json")
    with open(path, "w") as f:
        json.dump(stored, f)
    eng = Engine.__new__(Engine)
    eng.split_ways, eng.split_min, eng.split_rows = tune.tuned_engine(path)
    eng._split_stored = (eng.split_min, eng.split_rows)
    eng._split_rounds = tune.tuned_rounds(path)
    return eng


@pytest.mark.parametrize("rounds", ROUNDS)
def test_methods_with_rounds_keep_their_rule(tmp_path, rounds):
    from mpsim_amd.engine import SvdConfig
    eng = _engine(tmp_path, dict(split_ways=4, split_min=1, split_rows=257, split_min_rounds=2, split_rows_rounds=512))
    assert eng._split_rule(SvdConfig().to_c()) == (1, 257)
    assert eng._split_rule(SvdConfig(block=16, inner_sweeps=2).to_c()) == (1, 257)
    assert eng._split_rule(SvdConfig(**rounds).to_c()) == (2, 512)
    eng.split_min, eng.split_rows = 3, 100  # the caller's own
    assert eng._split_rule(SvdConfig(**rounds).to_c()) == (3, 100)


def test_one_rule_without_stored_rounds(tmp_path):
    from mpsim_amd.engine import SvdConfig
    eng = _engine(tmp_path, dict(split_ways=3, split_min=8, split_rows=128))
    assert eng._split_rule(SvdConfig(method=1).to_c()) == eng._split_rule(SvdConfig().to_c()) == (8, 128)


def test_repository_rule():
    from mpsim_amd import tune
    assert tune.tuned_rounds() == (2, 512)


@pytest.mark.parametrize("rows,fills", [([512] * 40, False), ([1024] * 3, False), ([1024] * 4, True), ([513] * 7, False),
                                        ([513] * 8, True), ([1040] * 9, False), ([1024] * 5 + [1040], False), ([1024, 1000, 900, 64], False)])
def test_calls_that_fill_the_device_stay_whole(rows, fills):
    """Groups of a workgroup for 16 rows, of problems of 513 to 1024 rows, on 256
    compute units."""
    from mpsim_amd.engine import Engine
    eng = Engine.__new__(Engine)
    eng._cus = 256
    assert eng._fills(rows) == fills
