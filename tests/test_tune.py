"""The tuner's choices (marvel_amd/tune.py) from given times; no GPU needed."""

import json

import pytest

from marvel_amd import tune
from marvel_amd.lib import lib


@pytest.fixture(autouse=True)
def defaults(monkeypatch, tmp_path):
    monkeypatch.setenv("MI_TUNE_CACHE", str(tmp_path))
    monkeypatch.setattr(tune, "device_key", lambda: "gfx950:256cu")
    yield
    lib.mi_set_tuning(None)


def test_a_level_without_tasks_keeps_its_default():
    """Every candidate of the wider levels reads 0 where no task gets there."""
    out = tune.tune_batch(lambda: [0, 0, int(1e6 / tune.current()["batch_waves_per_cu"]), 0, 0, 0, 0, 0])
    assert out["choice"]["batch_wide_waves_per_cu"] == tune.DEFAULT["batch_wide_waves_per_cu"]
    assert out["choice"]["batch_waves_per_cu"] == 24


@pytest.mark.parametrize("gain,want", [(0.01, 24), (0.1, 16)])
def test_a_candidate_has_to_be_faster_than_the_default_by_more_than_noise(gain, want):
    def run():
        t = 1.0 - gain if tune.current()["batch_waves_per_cu"] == 16 else 1.0
        return [0, 0, int(t * 1e6), 0, 0, 0, 0, 0]
    assert tune.tune_batch(run)["choice"]["batch_waves_per_cu"] == want


def test_report_shapes_keep_the_default_on_ties():
    out = tune.tune_report(lambda: ({"t_report_kernel": 0.5}, {"t_report_kernel": 0.5}))
    assert out["choice"] == {**out["choice"], "report_waves_per_cu": 24, "report_pool_log2": 15,
                             "report_l1_waves_per_cu": 8}


def test_a_choice_of_other_kernels_is_not_loaded(monkeypatch):
    tune.save(dict(tune.DEFAULT))
    assert tune.load_cached() == tune.DEFAULT
    with open(tune.cache_path()) as f:
        old = json.load(f)
    # as the earlier kernels stored theirs: by the device alone
    with open(tune.cache_path(), "w") as f:
        json.dump({tune.device_key(): {**tune.DEFAULT, "report_waves_per_cu": 32}}, f)
    assert tune.load_cached() is None
    with open(tune.cache_path(), "w") as f:
        json.dump(old, f)
    assert tune.load_cached() == tune.DEFAULT
    monkeypatch.setattr(tune, "GENERATION", tune.GENERATION + 1)
    assert tune.load_cached() is None
