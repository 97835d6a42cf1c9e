"""Partition of a search over tables under an estimate: what its scan batches left, or where a schedule of the DP
keeps none a run of its own; against the search over complete tables."""
import pytest

from tests.util import load_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule", ["", "history", "fused", "step"])
@pytest.mark.parametrize("plan, device", [(2, False), (3, False), (3, True)])
def test_partition_of_the_winner(monkeypatch, plan, device, schedule):
    from mist_amd.tune_one_case import PreparedSearch

    if device and schedule in ("history", "fused"):
        pytest.skip("one mesh for all stages: no such schedule")
    overrides = dict(tuning__tuning_granularity="uniform-device-pp") if device else {}
    search = PreparedSearch(load_plan(plan, model__num_hidden_layers=14, **overrides)[0])
    monkeypatch.setenv("MIST_DP_FORCE_SCHEDULE", schedule)
    stats = {}
    got = search.run(stats)
    assert got[1] is not None and not stats.get("stage_cost_cutoff_retries")
    monkeypatch.delenv("MIST_DP_FORCE_SCHEDULE")
    search.stage_cost_cutoff = None
    assert search.run() == got
