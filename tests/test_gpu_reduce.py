"""The pruned reduction against the kernel that evaluates every cell, at the edges of its tiles."""
import numpy as np
import pytest

from tests.util import assert_same_f64, tiny_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers, nodes, gpus, batch, samples, seeded", [
    (1, 1, 1, 2, 1, True),      # one layer: two pairs, one value of p
    (9, 1, 4, 16, 1, False),    # 54 pairs, empty minima at the start of the reduce launch
    (10, 1, 4, 16, 33, True),   # 65 pairs: a tile of one; a batch of 32 samples and one of 1
    (10, 1, 4, 16, 31, False),
    (66, 8, 8, 128, 1, True),   # 64 values of p: the minima of a pair are more than two per lane
    (66, 8, 8, 128, 5, True),
    (130, 2, 64, 128, 32, True),  # 128 of them: the samples of a pair do not fit the seeds' LDS at once
])
def test_pruned_tables_equal_every_cell_evaluated(layers, nodes, gpus, batch, samples, seeded, monkeypatch):
    import torch

    from mist_amd import intra_tuning
    from mist_amd.config import tp_candidates
    from mist_amd.intra_tuning import IntraStageTuner

    if not seeded:
        monkeypatch.setattr(intra_tuning, "SCOUT_MIN_STAGES", 0)
    cfg, tables = tiny_plan(1, layers=layers, hardware__num_nodes=nodes, hardware__num_gpus_per_node=gpus,
                            training__global_batch_size=batch, hardware__memory_capacity=8.0)
    devices = nodes * gpus
    meshes = [(1, 1)] if devices == 1 else [(1, 1), (1, 2), (nodes, gpus)]
    tp, Gs = tp_candidates(cfg)[0], [batch // 2, batch]
    got, want = [IntraStageTuner(tables, layers, meshes, Gs, tp, cfg, sample_size=samples, exhaustive=exhaustive).tune()
                 for exhaustive in (False, True)]
    finite = 0
    for v in range(4):
        for kind in ("index", "stable", "delta"):
            a, b = getattr(got.device, kind)[v], getattr(want.device, kind)[v]
            assert torch.equal(a, b), f"{kind} of variant {v}: {int((a != b).sum())} of {a.numel()} differ"
        finite += int(torch.isfinite(want.device.stable[v]).sum())
    assert finite > 0


@pytest.mark.parametrize("n_p, capacity, samples", [
    (2559, 90.0, 1), (2560, 90.0, 1),         # the minima of a pair in every wavefront's LDS, and not
    (10400, 300.0, 1), (10400, 300.0, 2),     # more than a workgroup's LDS: no seeds
    (36000, 1345.0, 1), (36000, 1345.0, 2),   # counts of more than 15 bits
])
def test_many_pre_saved_micro_batch_values(n_p, capacity, samples):
    """The stage operator takes the values of p from its caller."""
    from mist_amd.batched_module_analyzer import batched_tune_best_latency_for_stage as on_gpu
    from oracle.stage import batched_tune_best_latency_for_stage as on_cpu

    grid = [0.0, 0.5, 1.0]
    cfg, tables = tiny_plan(2, layers=2, hardware__num_nodes=1, hardware__num_gpus_per_node=2,
                            training__global_batch_size=16, hardware__memory_capacity=capacity,
                            tuning__search_space__offloading_ratio_candidates=grid,
                            tuning__search_space__sparse_offloading_ratio_candidates=grid)
    shape = (range(n_p), range(1, 3), range(3), 1, 2, 8)
    got = on_gpu(tables, None, None, *shape, cfg, tp_size=1, sample_size=samples)
    want = on_cpu(tables, cfg, *map(list, shape[:3]), *shape[3:], tp_size=1, sample_size=samples, inner="c")
    last = np.isfinite(want[0][0]).reshape(n_p, -1).any(axis=1).nonzero()[0].max()
    assert last > 0.6 * n_p, last
    for v in range(4):
        for i in range(3):
            assert_same_f64(got[v][i], want[v][i], f"result {i} of table {v}")


def test_more_than_65535_tiles_of_pairs():
    """2900 layers: 4.2e6 (l, c) pairs."""
    import torch

    from mist_amd.intra_tuning import IntraStageTuner

    layers = 2900
    cfg, tables = tiny_plan(2, layers=layers, hardware__num_nodes=1, hardware__num_gpus_per_node=2,
                            training__global_batch_size=4, hardware__memory_capacity=1500.0,
                            tuning__search_space__offloading_ratio_candidates=[0.0, 1.0],
                            tuning__search_space__sparse_offloading_ratio_candidates=[0.0, 1.0])
    got, want = [IntraStageTuner(tables, layers, [(1, 2)], [2], 1, cfg, sample_size=1, exhaustive=exhaustive).tune()
                 for exhaustive in (False, True)]
    for v in range(4):
        for kind in ("index", "stable", "delta"):
            a, b = getattr(got.device, kind)[v], getattr(want.device, kind)[v]
            assert torch.equal(a, b), f"{kind} of variant {v}: {int((a != b).sum())} of {a.numel()} differ"
    assert 0 < int(torch.isfinite(want.device.stable[0]).sum()) < want.device.stable[0].numel()
    assert bool(torch.isfinite(want.device.stable[0][0, 0, 0, 2890]).any())
