"""Cells that are in no pipeline below the limit are not looked for: the search over such tables returns what it
returns over complete ones."""
import numpy as np
import pytest

from tests.test_gpu_inter import _realistic_plan
from tests.util import load_plan

pytestmark = pytest.mark.gpu


def _stage_costs(search, cutoff):
    """The stage costs a search reads of the tables under ``cutoff`` (None: complete ones), per variant, the strategy
    rows, and per row of the tables the smallest largest stage cost of a pipeline."""
    from mist_amd import _lib, inter_tuning

    hw = search.config.hardware
    result = search.tuner.run_prepared(search.plan, search.dev_plan, cutoff)[0]
    uniform = None
    if search.granularity == "uniform-device-pp":
        uniform = dict(num_nodes=hw.num_nodes, num_gpus_per_node=hw.num_gpus_per_node,
                       ckpt_tuning=search.config.tuning.activation_checkpointing_tuning_enabled)
    runner = inter_tuning._DpRunner(result, search.L, hw.num_nodes * hw.num_gpus_per_node, search.meshes, 0, uniform)
    rows = np.arange(runner.Gn, dtype=np.int32)
    bottleneck = np.full(runner.Gn, np.inf, dtype=np.float32)
    for family in runner.families:
        found = runner.run(rows, np.zeros(runner.Gn, np.float32), _lib.DP_BOTTLENECK, family=family)
        bottleneck = np.minimum(bottleneck, np.where(found[0] >= 0, found[1], np.inf))
    return ([c.cpu().numpy() for c in runner.cost], [i[..., 0].cpu().numpy() for i in result.batch.index],
            bottleneck.astype(np.float64))


def _compare(cfg):
    """Cells that hold a row in the tables with closed cells and in those under the estimate alone.  Every threshold
    candidate that the search reads is in both."""
    from mist_amd import _lib
    from mist_amd.tune_one_case import PreparedSearch

    search = PreparedSearch(cfg)
    assert search.stage_cost_cutoff["close_unused"]
    got = search.run()
    estimate = search.dev_plan["incumbent"].item()
    full, rows, bottleneck = _stage_costs(search, None)
    closed, closed_rows, its_bottleneck = _stage_costs(search, search.stage_cost_cutoff)
    _, open_rows, _ = _stage_costs(search, dict(search.stage_cost_cutoff, close_unused=False))
    G = np.array(search.Gs * (len(bottleneck) // len(search.Gs)), dtype=np.float64)
    limit = estimate * (1.0 + _lib.load().mist_incumbent_slack()) * (1.0 - 1e-5) / G
    # (float32 costs against the bounds: a few units in the last place)
    reached = bottleneck <= np.minimum(limit, np.finfo(np.float32).max)
    least = np.where(reached, bottleneck, 0.0)
    least = least - 16.0 * (1e-4 + 1e-5 * least) + 1e-6 * least
    assert (its_bottleneck[reached] == bottleneck[reached]).all() and (its_bottleneck[~reached] >= limit[~reached]).all()
    n_closed = n_open = n_exact = 0
    for v in range(4):
        per_row = lambda x: x.reshape(-1, *[1] * (full[v].ndim - 1))
        exact = (full[v] >= per_row(least)) & (full[v] <= per_row(limit * (1.0 - 1e-6)))
        exact &= per_row(reached)
        assert (closed[v] >= full[v]).all()
        assert (closed[v][exact] == full[v][exact]).all() and (closed_rows[v][exact] == rows[v][exact]).all()
        # what else differs is no candidate of the search
        other = (closed[v] != full[v]) & per_row(reached)
        assert ((closed[v] < per_row(least)) | (closed[v] > per_row(limit * (1.0 - 1e-6))))[other].all()
        n_exact += int(exact.sum())
        n_closed, n_open = n_closed + int((closed_rows[v] >= 0).sum()), n_open + int((open_rows[v] >= 0).sum())
    assert n_exact > 0
    search.stage_cost_cutoff = None
    assert search.run() == got
    return n_closed, n_open, estimate


@pytest.mark.parametrize("plan, layers, nodes, batch, device", [
    (2, 32, 4, 512, False),   # the 7B plan
    (3, 37, 4, 256, True),    # uniform-device-pp, odd layers
    (3, 23, 5, 256, False),   # five nodes: no mesh of all devices
    (4, 20, 3, 768, False),
    (3, 9, 8, 512, False),    # fewer layers than stages of the smallest meshes
])
def test_search_over_tables_with_closed_cells(plan, layers, nodes, batch, device):
    overrides = dict(tuning__tuning_granularity="uniform-device-pp") if device else {}
    n_closed, n_open, _ = _compare(load_plan(plan, model__num_hidden_layers=layers, hardware__num_nodes=nodes,
                                          training__global_batch_size=batch, **overrides)[0])
    assert n_closed < n_open


@pytest.mark.parametrize("seed", [300000 + i for i in (
    0, 1, 3, 4, 6, 8, 10, 14, 15, 16, 17, 18, 19, 21, 23, 26, 27, 28, 30, 31, 34, 35, 36, 41, 46, 50, 55, 56, 57, 58,
    44)])  # (the last one: no estimate)
def test_random_plans_with_closed_cells(monkeypatch, seed):
    from mist_amd import intra_tuning

    monkeypatch.setattr(intra_tuning, "CLOSE_MIN_ITEMS", 0)  # (more than half of them are smaller)
    n_closed, n_open, estimate = _compare(_realistic_plan(seed))
    assert n_closed < n_open if estimate < float("inf") else n_closed == n_open
    assert (estimate < float("inf")) == (seed != 300044)


@pytest.mark.parametrize("plan, layers, memory, device", [
    (3, 37, 3.0, False), (3, 37, 4.0, False), (5, 79, 6.0, False), (3, 37, 3.0, True),
])
def test_tables_without_an_estimate_are_complete(plan, layers, memory, device):
    """Little memory and layers that no stage count divides: the only pipeline of equal stages is one on all devices,
    which does not fit, so there is no estimate though there are results.  What reads the tables takes them for
    complete then: no cell is closed (one of the mesh of all devices would be, whose layers are not all there are)."""
    from mist_amd.tune_one_case import PreparedSearch

    overrides = dict(tuning__tuning_granularity="uniform-device-pp") if device else {}
    search = PreparedSearch(load_plan(plan, model__num_hidden_layers=layers, hardware__num_nodes=4 if plan == 3 else 8,
                                      training__global_batch_size=256, hardware__memory_capacity=memory, **overrides)[0])
    cost, solution = search.run()
    assert solution is not None and search.dev_plan["incumbent"].item() == float("inf")
    closed = search.tuner.run_prepared(search.plan, search.dev_plan, search.stage_cost_cutoff)[0].batch
    without = dict(search.stage_cost_cutoff, close_unused=False)
    open_ = search.tuner.run_prepared(search.plan, search.dev_plan, without)[0].batch
    for v in range(4):
        has = open_.index[v] >= 0
        assert bool((closed.index[v] == open_.index[v]).all())
        for ours, theirs in ((closed.stable, open_.stable), (closed.delta, open_.delta)):
            assert bool((ours[v][has] == theirs[v][has]).all())
    search.stage_cost_cutoff = None
    assert search.run() == (cost, solution)


@pytest.mark.parametrize("dense", [False, True])
def test_windows_that_reach_below_what_such_tables_hold(dense):
    """A window whose threshold candidates have no certain start within two widenings (values half a gap apart, in
    cells of a mesh of all devices that no pipeline uses) leaves the search undecided."""
    import torch

    from mist_amd import _lib, inter_tuning
    from tests.test_gpu_inter import _synthetic_results

    L, D, Gs, meshes = 20, 16, [2], [(1, 1), (1, 2), (1, 4), (2, 4), (4, 4)]
    (ours,), _ = _synthetic_results(np.random.default_rng(5), 1, Gs, meshes, L, 16, 1, 1 / 256, 0.1, structured=True,
                                    structured_exponent=1.0, jitter=0.0)
    runner = inter_tuning._DpRunner(ours, L, D, meshes, 0)
    _, bottleneck, _ = runner.run(np.zeros(1, np.int32), np.zeros(1, np.float32), _lib.DP_BOTTLENECK)
    tables = ours.device
    if dense:
        cells = [(p, l, c) for p in range(16) for l in range(2, L - 1) for c in range(l + 1) if c != l - 1 or p == 0]
        where = torch.tensor(cells, device="cuda").T
        values = float(bottleneck[0]) - 9e-7 * torch.arange(1, 2 * len(cells) + 1, device="cuda", dtype=torch.float64)
        # further than sixteen times the first margin
        assert 9e-7 * len(values) > 16 * (1e-4 + 1e-5 * float(bottleneck[0])) * 1.1
        for v in range(2):  # base and with_pre
            at = (0, 4, where[0], where[1] - 1, where[2], 0)
            tables.stable[v][at], tables.delta[v][at] = values[v::2], 0.0
            tables.index[v][at] = 0
    limit = torch.full((1,), 1e3, dtype=torch.float64).pin_memory()
    stats = {}
    inter_tuning.inter_stage_tune_batch(L, D, meshes, Gs, [ours], slot=0, stats=stats, only_best_solution=True,
                                        table_limit=(limit, 1.0))
    assert (stats["dp_undecided"] > 0) == dense
