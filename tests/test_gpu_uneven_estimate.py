"""Estimate of the cost of the best pipeline where the stages of a mesh do not divide the layers."""
import numpy as np
import pytest

from tests.util import load_plan

pytestmark = pytest.mark.gpu


def _best_pipeline(full, Gs, meshes, L, D):
    """Cheapest pipeline of S = D / (n m) stages on one mesh that the finished tables hold, with L // S
    layers a stage and one more in the first L % S stages behind the first one."""
    best = float("inf")
    tables = [(full.stable[v][..., 0].cpu().numpy(), full.delta[v][..., 0].cpu().numpy(), full.index[v][..., 0].cpu().numpy())
              for v in range(4)]
    for row in range(tables[0][0].shape[0]):
        G = Gs[row % len(Gs)]
        for q, (n, m) in enumerate(meshes):
            S = D // (n * m)
            if D % (n * m) or S > L or S - 1 >= tables[0][0].shape[2] or S > min(D, L) // 2:
                continue
            costs, end = [], -1
            for s in range(S):
                l = L // S + (1 if 1 <= s <= L % S else 0)
                end += l
                v = 3 if S == 1 else 1 if s == 0 else 2 if s == S - 1 else 0
                cell = (row, q, S - 1 - s, l - 1) if v < 2 else (row, q, l - 1)
                stable, delta, index = (t[cell] for t in tables[v])
                cost = stable + (np.float32(delta) / np.float32(G) if v == 0 else delta / G)
                costs.append(np.where(index >= 0, cost, np.inf)[:min(l, L - end) + 1].min())
            assert end == L - 1
            if np.isfinite(costs).all():
                best = min(best, sum(costs) + (G - 1) * max(costs))
    return best


@pytest.mark.parametrize("plan, layers, nodes, batch", [
    (3, 23, 5, 256),   # five stages of 4, 5, 5, 5, 4 layers, ten of 2 and 3; no mesh has stages that divide both
    (4, 20, 3, 768),   # three of 6, 7, 7: the last one with the extra layer
    (3, 16, 6, 96),    # three of 5, 6, 5; more stages on the smallest meshes than layers
])
def test_pipelines_with_an_uneven_number_of_layers(plan, layers, nodes, batch):
    """The estimate exists, is no smaller than the best such pipeline of the complete tables (it is one
    made of some rows), and ``tune`` returns what it returns without it."""
    from mist_amd.tune_one_case import PreparedSearch

    cfg, _ = load_plan(plan, model__num_hidden_layers=layers, hardware__num_nodes=nodes, training__global_batch_size=batch)
    search = PreparedSearch(cfg)
    D = cfg.hardware.num_nodes * cfg.hardware.num_gpus_per_node
    full = search.tuner.run_prepared(search.plan, search.dev_plan)[0].batch
    in_tables = _best_pipeline(full, search.Gs, search.tuner.device_mesh_candidates, layers, D)
    got = search.run()
    estimate = float(search.dev_plan["incumbent"].item())
    assert np.isfinite(estimate) and np.isfinite(in_tables)
    assert estimate >= in_tables * (1.0 - 1e-12)  # (a sum of at most L float64 terms in another order)
    search.stage_cost_cutoff = None
    assert search.run() == got
