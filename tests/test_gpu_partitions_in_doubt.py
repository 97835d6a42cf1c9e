"""Partitions that tables under an estimate leave in doubt: settled by the search where the result is the same
whether the reference finds them or not, by a second evaluation on complete tables elsewhere."""
import pytest

from tests.test_gpu_inter import _realistic_plan, _sparse_candidate_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed, evaluations", [
    (3, 0),          # of the instance of the result: the scan ends the same either way
    (252, 0), (499, 0), (200146, 0),
    (200117, 0),     # two
    (785, 1), (972, 1), (823, 1),  # cheaper than what the scan found
    (None, 1),       # it is what the reference returns
])
def test_result_is_that_of_complete_tables(seed, evaluations):
    from mist_amd.tune_one_case import PreparedSearch

    search = PreparedSearch(_sparse_candidate_plan() if seed is None else _realistic_plan(seed))
    stats = {}
    got = search.run(stats)
    assert stats["dp_unresolved"] > 0 and stats.get("stage_cost_cutoff_retries", 0) == evaluations
    assert stats.get("stage_cost_doubts_settled", 0) == 1 - evaluations
    search.stage_cost_cutoff = None
    assert search.run() == got
