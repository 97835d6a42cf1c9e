"""The cost table kernels at the row lengths where their shifts, their workgroups and their passes end."""
import numpy as np
import pytest

import tests.test_gpu_inter as inter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L, P1", [(15, 2), (16, 2), (31, 2), (63, 2), (64, 2), (127, 2), (128, 2), (255, 2),
                                   (256, 2), (257, 2)])
def test_cost_tables_at_the_edges_of_a_row(L, P1):
    inter.test_cost_tables_and_running_minima_equal_numpy(L, P1, 1 / 8, 0.4)


@pytest.mark.parametrize("L, P1", [(2, 3), (3, 5), (4, 2), (15, 2), (62, 2), (63, 2), (64, 3), (80, 2), (127, 2),
                                   (128, 3), (254, 2), (255, 2), (256, 2)])
def test_cost_tables_of_one_sample(L, P1):
    """Four cells a lane: sets of rows that cross a gradient accumulation, the last cells of a table, rows
    over two wavefronts, cells without a strategy whose costs are not read."""
    import torch

    from mist_amd.inter_tuning import _DpRunner

    rng = np.random.default_rng(L)
    meshes, Gs = [(1, 1), (1, 2), (1, 4)], [1, 3, 8]
    ours, theirs = inter._synthetic_results(rng, 2, Gs, meshes, L, P1, 1, 1 / 1024, 0.6, structured=False)
    names = ("costs_stable", "costs_stable_with_pre", "costs_stable_with_post", "costs_stable_no_pp")
    runner = _DpRunner(ours[0], L, 4, meshes, 0)
    costs = [t.clone() for t in runner.cost], [t.clone() for t in runner.pmin]
    whole = ours[0].batch
    for v in range(4):
        whole.stable[v][whole.index[v] < 0] = 0.0
    runner = _DpRunner(ours[0], L, 4, meshes, 0)
    for kind, want in zip((runner.cost, runner.pmin), costs):
        assert all(torch.equal(a, b) for a, b in zip(kind, want))
    G_of_row = np.tile(np.array(Gs, dtype=np.float32), 2)
    for v, name in enumerate(names):
        stable = np.concatenate([getattr(t, name)[..., 0] for t in theirs])
        delta = np.concatenate([getattr(t, name.replace("stable", "delta"))[..., 0] for t in theirs])
        with np.errstate(invalid="ignore"):
            want = (stable + delta / G_of_row.reshape((-1,) + (1,) * (stable.ndim - 1))).astype(np.float32)
        assert np.array_equal(costs[0][v].cpu().numpy().view(np.int32), want.view(np.int32)), name
        want_min = np.minimum.accumulate(want, axis=-1)
        assert np.array_equal(costs[1][v].cpu().numpy().view(np.int32), want_min.view(np.int32)), name
