"""Tables of which only some planes of the p axis are filled, against complete ones: cost tables, re-laid row
minima, threshold candidates, the searches, and ``tune`` on memory full of other values."""
import numpy as np
import pytest

import tests.test_gpu_inter as inter

pytestmark = pytest.mark.gpu


def _unwritten(L, P1, v):
    """Cells of a (row of the tables, mesh) that no plan writes (batched_module_analyzer.py:3021-3023, 3103)."""
    l, c = np.arange(1, L + 1)[:, None], np.arange(L + 1)[None, :]
    if v == 3:
        return np.arange(L + 1) == L - 1
    if v == 2:
        return (c > l) | (c == l - 1)
    return np.stack([(c > l) | ((c == l - 1) & (p > 0)) for p in range(P1)])


@pytest.mark.parametrize("L, P1, meshes", [
    (2, 2, [(1, 1), (1, 2)]), (5, 4, [(1, 1), (1, 2), (1, 4)]), (15, 6, [(1, 1), (1, 2), (1, 4)]),
    (32, 5, [(1, 1), (1, 2), (1, 4), (1, 8)]), (80, 9, [(1, 1), (1, 2), (1, 4)]), (180, 3, [(1, 2), (1, 4)]),
    (181, 3, [(1, 2), (1, 4)]), (255, 2, [(1, 2), (1, 4)]),
])
def test_planes_equal_complete_tables(L, P1, meshes):
    import torch

    from mist_amd.inter_tuning import _DpRunner, inter_stage_tune_batch

    rng = np.random.default_rng(L + 31 * P1)
    Gs, entries = [1, 4, 16], 2
    ours, _ = inter._synthetic_results(rng, entries, Gs, meshes, L, P1, 1, 1 / 1024, 0.3, structured=True)
    whole = ours[0].batch
    Gn, Q = entries * len(Gs), len(meshes)
    planes = rng.integers(0, P1 + 1, size=(Gn, Q)).astype(np.int32)
    planes[0, 0], planes[-1, -1] = 0, P1
    planes[2, -1], planes[3, 0] = P1 + 3, -2  # (as P1 and 0)
    missing = []
    for v in range(4):
        gone = np.broadcast_to(_unwritten(L, P1, v), whole.index[v].shape[:-1]).copy()
        if v < 2:
            gone |= (np.arange(P1) >= planes[:, :, None])[..., None, None]
        else:
            gone[planes <= 0] = True
        missing.append(torch.from_numpy(gone).cuda()[..., None])
        whole.index[v][missing[v]] = -1
        whole.stable[v][missing[v]] = float("inf")
        whole.delta[v][missing[v]] = float("inf")
    D = max(n * m for n, m in meshes)

    def everything():
        runner = _DpRunner(ours[0], L, D, meshes, 0)
        rows = np.arange(Gn, dtype=np.int32)
        lo, hi = np.full(Gn, -np.inf, np.float32), np.linspace(0.5, 2.0, Gn).astype(np.float32) * L
        lo[1], hi[1] = np.inf, np.inf  # (nothing feasible)
        values, bounds, above = runner.candidates_between_flat(rows, lo, hi)
        return runner, (values.tolist(), bounds.tolist(), above.tolist())

    full, want_candidates = everything()
    uniform = dict(num_nodes=1, num_gpus_per_node=D, ckpt_tuning=True)
    searches = [None] + ([uniform] if (1, 1) in meshes else [])
    want = [inter_stage_tune_batch(L, D, meshes, Gs, ours, uniform_device=u) for u in searches]
    # what is not there may hold anything
    whole.planes = torch.from_numpy(planes).cuda()
    for v in range(4):
        whole.index[v][missing[v]] = 3
        whole.stable[v][missing[v]] = 1e-3
        whole.delta[v][missing[v]] = 1e-3
        none = (whole.index[v] < 0)
        whole.stable[v][none] = 1e-3
        whole.delta[v][none] = 1e-3
    some, got_candidates = everything()
    held = torch.from_numpy(np.arange(P1) < planes[:, :, None]).cuda()
    for kind in ("cost", "pmin"):
        for v in range(4):
            a, b = getattr(full, kind)[v], getattr(some, kind)[v]
            keep = held if v < 2 else whole.planes > 0
            assert torch.equal(a[keep], b[keep]), (kind, v)
    # (the stage up to the last layer is the last one: what its entries hold for p > 0 is never read)
    S = full.families[0].S_max
    starts = np.cumsum([0] + [L - k for k in range(L)])
    last = torch.from_numpy(starts[1:] - 1).cuda()
    minima = [r.families[0].stage_min.view(Gn, S, Q, -1) for r in (full, some)]
    for m in minima:
        m[:, 1:, :, last] = float("inf")
    assert torch.equal(*minima)
    assert got_candidates == want_candidates
    assert [inter_stage_tune_batch(L, D, meshes, Gs, ours, uniform_device=u) for u in searches] == want


def _leave_used_memory(value):
    """Blocks of the allocator's two pools that hold ``value`` and are free again."""
    import torch

    torch.cuda.empty_cache()
    used = [torch.full((1 << bits,), value, dtype=torch.int32, device="cuda")
            for bits in [28, 26, 24, 22, 20] + [bits for bits in range(18, 6, -1) for _ in range(48)]]
    del used


def _count_used_tables(monkeypatch, tuner, value):
    """How often the tables of ``tuner`` begin as indices of ``value`` and nothing else."""
    import torch

    allocate, seen = tuner._allocate_flat, []

    def allocated(*args):
        costs, index, struct = allocate(*args)
        seen.append(torch.equal(index, torch.full_like(index, value)))
        return costs, index, struct

    monkeypatch.setattr(tuner, "_allocate_flat", allocated)
    return seen


@pytest.mark.parametrize("granularity", ["inter-stage", "uniform-device-pp"])
def test_tune_on_used_memory(monkeypatch, granularity):
    """Tables that nothing fills lie in memory that held other indices and costs."""
    from mist_amd.tune_one_case import PreparedSearch
    from tests.util import load_plan

    cfg, _ = load_plan(1, tuning__tuning_granularity=granularity)
    want = PreparedSearch(cfg).run()
    for value in (0, 5, 0x3f000000):
        search = PreparedSearch(cfg)
        seen = _count_used_tables(monkeypatch, search.tuner, value)
        _leave_used_memory(value)
        assert search.run() == want
        assert seen and seen[0], value


@pytest.mark.parametrize("native", [True, False])
def test_parts_of_a_run_without_a_fill(monkeypatch, native):
    """A search over some tensor-parallel candidates of such a run, and tables read from its results, know which
    cells hold something too."""
    import mist_amd.inter_tuning as inter_tuning
    from mist_amd.intra_tuning import VARIANTS, IntraStageTunerOutput
    from mist_amd.tune_one_case import PreparedSearch
    from tests.util import load_plan

    monkeypatch.setattr(inter_tuning, "NATIVE_SEARCH", native)
    cfg, _ = load_plan(2)
    search = PreparedSearch(cfg)
    hw = cfg.hardware
    find = lambda results: inter_tuning.inter_stage_tune_batch(
        search.L, hw.num_nodes * hw.num_gpus_per_node, search.meshes, search.Gs, results)
    complete = search.tuner.run_prepared(search.plan, search.dev_plan)
    want = find(complete)
    assert len(want) > 2 and sum(solution is not None for _, solution in want) > 1
    seen = _count_used_tables(monkeypatch, search.tuner, 7)
    run = lambda: search.tuner.run_prepared(search.plan, search.dev_plan, fill_costs=False, sparse=True)
    _leave_used_memory(7)
    results = run()
    assert seen[0] and results[0].batch.planes is not None
    assert find(results) == want
    assert find(results[1:]) == want[1:]  # (their own tables, cut out of the batch)
    other = run()
    assert find([results[0], other[1]]) == want[:2]
    for t, (a, b) in enumerate(zip(run(), complete)):
        assert np.array_equal(a.device.grad_accum.cpu().numpy(), search.Gs)
        for v, suffix in enumerate(VARIANTS):
            for kind in ("indices", "costs_stable", "costs_delta"):
                assert np.array_equal(getattr(a, kind + suffix), getattr(b, kind + suffix)), (t, v, kind)
    some = run()[1]
    cells = [(0, 0, 1, 3, 3, 0), (1, 1, 0, 0, 1, 0), (0, 1, 0, 4, 2, 0)]
    for a, b in zip(IntraStageTunerOutput.solutions_at([(some, 0, cell) for cell in cells]),
                    IntraStageTunerOutput.solutions_at([(complete[1], 0, cell) for cell in cells])):
        assert np.array_equal(a, b)
