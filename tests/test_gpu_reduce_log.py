"""The log of rows that reached a minimum: none, one that runs full (the opened items are gone through again), a
whole one; against the kernel that evaluates every cell."""
import pytest

from tests.util import tiny_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", ["0", "1", "7", ""])
@pytest.mark.parametrize("samples, seeded", [(1, True), (1, False), (3, True), (30, False)])
def test_rows_of_the_minima(monkeypatch, samples, seeded, chunks):
    import torch

    from mist_amd import intra_tuning
    from mist_amd.config import tp_candidates
    from mist_amd.intra_tuning import IntraStageTuner

    monkeypatch.setenv("MIST_REDUCE_LOG_CHUNKS", chunks)
    if not seeded:
        monkeypatch.setattr(intra_tuning, "SCOUT_MIN_STAGES", 0)
    cfg, tables = tiny_plan(2, layers=13, hardware__num_nodes=2, hardware__num_gpus_per_node=4,
                            training__global_batch_size=48, hardware__memory_capacity=9.0)
    tp, meshes = tp_candidates(cfg)[0], [(1, 1), (1, 4), (2, 4)]
    got, want = [IntraStageTuner(tables, 13, meshes, [3, 6, 24], tp, cfg, sample_size=samples, exhaustive=exhaustive).tune()
                 for exhaustive in (False, True)]
    assert any(int((index >= 0).sum()) for index in want.device.index)
    for v in range(4):
        for kind in ("index", "stable", "delta"):
            a, b = getattr(got.device, kind)[v], getattr(want.device, kind)[v]
            assert torch.equal(a, b), f"{kind} of variant {v}: {int((a != b).sum())} of {a.numel()} differ"
