"""Several uniform-device families in one launch against a launch for each and, where its interpreted loops
allow, the oracle."""
import numpy as np
import pytest

import tests.test_gpu_inter as inter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes, gpus, n_families", [(1, 1, 1), (4, 2, 4), (24, 4, 8), (36, 2, 9)])
def test_families_of_one_launch_equal_single_ones(monkeypatch, nodes, gpus, n_families):
    """Up to as many as a launch takes and one more; the python driver runs them one by one."""
    from mist_amd import inter_tuning
    from mist_amd.inter_tuning_uniform import _uniform_device_mesh_partition

    L = max(min(nodes * gpus, 36), 2)
    meshes = sorted({mesh for S in range(1, L + 1) if (mesh := _uniform_device_mesh_partition(S, nodes, gpus))})
    assert len(meshes) == n_families
    ours, theirs = inter._synthetic_results(np.random.default_rng(nodes), 2, [1, 4], meshes, L, L, 1, 1 / 64, 0.3,
                                            structured=True)
    uniform = dict(num_nodes=nodes, num_gpus_per_node=gpus, ckpt_tuning=True)
    found = []
    for native in (True, False):
        monkeypatch.setattr(inter_tuning, "NATIVE_SEARCH", native)
        found.append(inter_tuning.inter_stage_tune_batch(L, nodes * gpus, meshes, [1, 4], ours, stats={},
                                                         uniform_device=uniform))
    assert found[0] == found[1]
    assert any(solution is not None for _, solution in found[0])
    if nodes * gpus <= 8:
        from oracle import inter_uniform_device

        class Config:
            class tuning:
                activation_checkpointing_tuning_enabled = True

        assert found[0] == [inter_uniform_device.inter_stage_tune(L, nodes, gpus, meshes, [1, 4], r, Config)
                            for r in theirs]
