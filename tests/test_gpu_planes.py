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
    missing = []
    for v in range(4):
        gone = np.broadcast_to(_unwritten(L, P1, v), whole.index[v].shape[:-1]).copy()
        if v < 2:
            gone |= (np.arange(P1) >= planes[:, :, None])[..., None, None]
        else:
            gone[planes == 0] = True
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


@pytest.mark.parametrize("granularity", ["inter-stage", "uniform-device-pp"])
def test_tune_on_used_memory(granularity):
    """Tables that nothing fills lie in memory that held other indices and costs."""
    import torch

    from mist_amd.tune_one_case import PreparedSearch
    from tests.util import load_plan

    cfg, _ = load_plan(1, tuning__tuning_granularity=granularity)
    want = PreparedSearch(cfg).run()
    for value in (0, 5, 0x3f000000):
        torch.cuda.empty_cache()
        used = [torch.full((n,), value, dtype=torch.int32, device="cuda") for n in (1 << 20, 1 << 24, 1 << 26)]
        del used
        assert PreparedSearch(cfg).run() == want
