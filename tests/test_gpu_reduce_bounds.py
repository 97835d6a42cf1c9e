"""The reduction's bounds against the kernel that evaluates every cell, where memory decides."""
import pytest

from tests.test_gpu_reduce import test_many_pre_saved_micro_batch_values as hold_against_the_oracle
from tests.util import tiny_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_p", [2543, 2544])
def test_minima_and_candidates_in_lds(n_p):
    """As many values of p as a workgroup's LDS holds beside the lists of candidates, and one more."""
    hold_against_the_oracle(n_p, 90.0, 1)


@pytest.mark.parametrize("samples", [1, 2, 7, 32])
@pytest.mark.parametrize("base, capacity", [(1, 3.0), (1, 3.9), (1, 5.0), (2, 9.0), (2, 12.0), (2, 20.0)])
def test_where_memory_decides(base, capacity, samples):
    """From plans of which a few cells fit to plans with most of them: counts at their edges, last and
    single stages that just fit, pairs without any minimum; G that is no power of two."""
    import torch

    from mist_amd.config import tp_candidates
    from mist_amd.intra_tuning import IntraStageTuner

    layers, meshes = 13, [(1, 1), (1, 4), (2, 4)]
    cfg, tables = tiny_plan(base, layers=layers, hardware__num_nodes=2, hardware__num_gpus_per_node=4,
                            training__global_batch_size=48, hardware__memory_capacity=capacity)
    finite = 0
    for tp in tp_candidates(cfg)[:2]:
        got, want = [IntraStageTuner(tables, layers, meshes, [3, 6, 24], tp, cfg, sample_size=samples,
                                     exhaustive=exhaustive).tune() for exhaustive in (False, True)]
        for v in range(4):
            for kind in ("index", "stable", "delta"):
                a, b = getattr(got.device, kind)[v], getattr(want.device, kind)[v]
                assert torch.equal(a, b), f"tp {tp}, {kind} of variant {v}: {int((a != b).sum())} of {a.numel()} differ"
            finite += int(torch.isfinite(want.device.stable[v]).sum())
    assert finite > 0
