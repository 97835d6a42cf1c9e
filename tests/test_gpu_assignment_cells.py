"""Layer counts that are in no assignment near the estimate of the best are left out of the tables: ``tune`` returns
what it returns over complete ones, and evaluates again where the optimum is above the estimate."""
import pytest

from tests.util import load_plan

pytestmark = pytest.mark.gpu


def _plan(plan, layers, nodes, batch, tuned, samples=30):
    return load_plan(plan, model__num_hidden_layers=layers, hardware__num_nodes=nodes, training__global_batch_size=batch,
                     tuning__tuning_granularity="uniform-device-pp-mip", tuning__sample_size=samples,
                     tuning__activation_checkpointing_tuning_enabled=tuned)[0]


def _cells_with_a_row(monkeypatch):
    """How many cells of the tables hold a row, call by call."""
    from mist_amd import intra_tuning

    run, held = intra_tuning.IntraStageTuner.run_prepared, []

    def counted(tuner, *args, **kwargs):
        out = run(tuner, *args, **kwargs)
        wanted = tuner._plan["wanted"]
        n = 0
        for g, q in zip(*(wanted[:, :, 0] >= 0).nonzero()):
            first, last, planes = (int(x) for x in wanted[g, q, :3])
            n += int((out[0].batch.index[2][g::wanted.shape[0], q, first - 1:last] >= 0).sum())
        held.append(n)
        return out

    monkeypatch.setattr(intra_tuning.IntraStageTuner, "run_prepared", counted)
    return held


@pytest.mark.parametrize("plan, layers, nodes, batch, tuned, samples", [
    (2, 32, 4, 512, True, 30),
    (2, 17, 2, 64, True, 7),     # layers that no stage count divides
    (2, 13, 1, 8, False, 30),    # every layer checkpointed
    (3, 9, 4, 256, True, 33),    # more samples than one set of launches takes
    (3, 23, 5, 256, True, 2),    # five nodes
    (3, 2, 1, 16, True, 3),
])
def test_assignment_over_the_cells_left(monkeypatch, plan, layers, nodes, batch, tuned, samples):
    from mist_amd import _lib, intra_tuning
    from mist_amd.tune_one_case import tune

    monkeypatch.setattr(intra_tuning, "ASSIGNMENT_MIN_ITEMS", 0)
    cfg = _plan(plan, layers, nodes, batch, tuned, samples)
    held = _cells_with_a_row(monkeypatch)
    stats = {}
    got = tune(cfg, stats=stats)
    monkeypatch.setenv("MIST_NO_STAGE_COST_CUTOFF", "1")
    want = tune(cfg)
    assert got == want and "mip_second_evaluations" not in stats
    assert sum(held[:len(held) // 2]) < sum(held[len(held) // 2:])
    assert want[1] is None or stats["mip_estimate"] > 0
    # an optimum that is not below the estimate's room: the second evaluation
    monkeypatch.delenv("MIST_NO_STAGE_COST_CUTOFF")
    monkeypatch.setattr(_lib.load(), "mist_incumbent_slack", lambda: -0.5)
    stats = {}
    assert tune(cfg, stats=stats) == want
    assert want[1] is None or stats["mip_second_evaluations"] == 1
