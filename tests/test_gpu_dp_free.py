"""The recurrence of one mesh for all stages in one workgroup against a launch per stage count, at the layer counts
where the values that a thread reads ahead, and the eight lanes of a start layer, begin and end."""
import numpy as np
import pytest

import tests.test_gpu_inter as inter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ckpt_tuning", [True, False])
@pytest.mark.parametrize("L, nodes, gpus", [
    (1, 1, 1), (2, 1, 2), (7, 1, 4), (8, 2, 4), (9, 2, 4), (22, 8, 2), (23, 2, 8), (45, 4, 8), (46, 4, 8), (63, 2, 8),
    (64, 2, 8), (90, 1, 8), (91, 1, 8), (110, 1, 4),
])
def test_one_workgroup_equals_a_launch_per_stage_count(monkeypatch, L, nodes, gpus, ckpt_tuning):
    from mist_amd import _lib
    from mist_amd.inter_tuning import _DpRunner
    from mist_amd.inter_tuning_uniform import _uniform_device_mesh_partition

    D = nodes * gpus
    meshes = sorted({mesh for S in range(1, L + 1) if (mesh := _uniform_device_mesh_partition(S, nodes, gpus))})
    P1 = min(D, L)
    rng = np.random.default_rng(L)
    ours, _ = inter._synthetic_results(rng, 1, [2, 4], meshes, L, P1, 1, 1 / 64, 0.3, structured=True)
    runner = _DpRunner(ours[0], L, D, meshes, 0, dict(num_nodes=nodes, num_gpus_per_node=gpus, ckpt_tuning=ckpt_tuning))
    rows = np.array([0, 1, -1, 1, 0, 1], dtype=np.int32)
    feasible = 0
    for family in runner.families:
        _, bottleneck, _ = runner.run(rows, np.zeros(6, np.float32), _lib.DP_BOTTLENECK, family=family)
        t = np.where(np.isfinite(bottleneck), bottleneck, 1.0) * np.array([1, 1, 1, 1.1, 1.5, 9], np.float32)
        for mode in (_lib.DP_BOTTLENECK, _lib.DP_THRESHOLD):
            found = []
            for schedule in ("", "step"):
                monkeypatch.setenv("MIST_DP_FORCE_SCHEDULE", schedule)
                found.append(runner.run(rows, t.astype(np.float32), mode, family=family)[:3])
            for a, b in zip(*found):
                assert np.array_equal(a[rows >= 0], b[rows >= 0]), (family.S_max, mode)
            feasible += int((found[0][0] > 0).sum())
    assert feasible > 0
