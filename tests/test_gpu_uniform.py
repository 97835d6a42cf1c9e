"""The uniform search on the device (``mist_uniform_search``) against the host loops over the same
tables, and ``tune`` over the cells it reads against the search over whole tables."""
import pytest

from tests.util import tiny_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers, nodes, gpn, samples, overrides", [
    (6, 2, 4, 1, dict()),
    (7, 2, 4, 30, dict()),                                                   # uneven layers, slot 0 of 30
    (9, 1, 8, 2, dict(tuning__activation_checkpointing_tuning_enabled=False)),
    (5, 2, 2, 30, dict(tuning__tuning_granularity="uniform-pp-simple-heuristic-mem-opt")),
    (4, 4, 2, 1, dict(hardware__memory_capacity=0.2)),                       # nothing fits
])
def test_device_search_equals_the_host_loops(layers, nodes, gpn, samples, overrides):
    from mist_amd.inter_tuning_uniform import _inter_stage_tune_on_host, inter_stage_tune
    from mist_amd.intra_tuning import IntraStageTuner
    from mist_amd.search_space import _get_device_mesh_candidates, _get_grad_accumu_steps_candidates
    from mist_amd.tune_one_case import PreparedSearch

    base = dict(hardware__num_nodes=nodes, hardware__num_gpus_per_node=gpn, hardware__memory_capacity=6.0,
                training__global_batch_size=32, tuning__tuning_granularity="uniform-pp")
    cfg, tables = tiny_plan(1, layers=layers, **{**base, **overrides})
    meshes = _get_device_mesh_candidates(nodes, gpn, False)
    Gs = _get_grad_accumu_steps_candidates(32)
    best = (float("inf"), None)
    for tp in (t for t in (1, 2, 4, 8) if t <= gpn):
        slots = [0] if samples > 1 else None
        res = IntraStageTuner(tables, layers, meshes, Gs, tp, cfg, sample_size=samples, sample_slots=slots).tune()
        got = inter_stage_tune(layers, nodes, gpn, Gs, res, cfg)
        assert got == _inter_stage_tune_on_host(layers, nodes, gpn, Gs, res, cfg)
        assert inter_stage_tune(layers, nodes, gpn, Gs[1:3], res, cfg) == _inter_stage_tune_on_host(
            layers, nodes, gpn, Gs[1:3], res, cfg)
        best = got if got[0] < best[0] else best
    if samples == 30:  # what tune() evaluates: the default number of samples, slot 0
        assert PreparedSearch(cfg).run() == best
