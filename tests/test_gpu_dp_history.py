"""The DP schedules that keep every plane and look winners up on the answer's path
(``dp_history_kernel``, ``dp_free_kernel``) against the one-launch-per-stage-count schedule, bit by bit."""
import ctypes
import os

import numpy as np
import pytest

from tests.test_gpu_inter import _random_tables

pytestmark = pytest.mark.gpu


def _run(meshes, L, D, P1, S, rule, tabs, g_index, tmax, mode, schedule, free=False, want_path=False):
    import torch

    from mist_amd import _lib

    lib = _lib.load()
    Q, n = len(meshes), len(tmax)
    shape = np.zeros(1, dtype=_lib.DP_SHAPE_DTYPE)
    shape["num_layers"], shape["num_devices"], shape["num_mesh"], shape["p_dim"] = L, D, Q, P1
    shape["max_stages"], shape["ckpt_rule"] = S, rule
    shape["free_devices"] = free
    shape["mesh_n"][0, :Q] = [a for a, _ in meshes]
    shape["mesh_m"][0, :Q] = [b for _, b in meshes]
    sp = ctypes.c_void_p(shape.ctypes.data)
    dev = [torch.from_numpy(np.stack([t[v] for t in tabs])).cuda() for v in range(4)]
    dev += [torch.cummin(t, dim=-1).values.contiguous() for t in dev]
    costs = _lib.DpCosts(*[t.data_ptr() for t in dev])
    for v in range(4):
        costs.g_stride[v] = dev[v][0].numel()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    per_g = lib.mist_dp_stage_minima_floats(sp)
    stage_min = torch.empty(per_g * len(tabs), dtype=torch.float32).cuda()
    _lib.check(lib.mist_dp_stage_minima(sp, ctypes.byref(costs), len(tabs), stage_min.data_ptr(), stream),
               "mist_dp_stage_minima")
    costs.stage_min, costs.stage_min_g_stride = stage_min.data_ptr(), per_g
    d_t = torch.tensor(np.asarray(tmax, dtype=np.float32)).cuda()
    d_g = torch.tensor(np.asarray(g_index, dtype=np.int32)).cuda()
    out = torch.full((3, n), -9.0, dtype=torch.float32).cuda()
    path = torch.full((n, S, 4), -9, dtype=torch.int32).cuda()
    argmin = torch.empty((n, S + 1, L + 1, D + 1, 4), dtype=torch.int32).cuda()
    floats = lib.mist_dp_scratch_floats_sized(sp, n)
    scratch = torch.empty(floats, dtype=torch.float32).cuda()
    old = os.environ.get("MIST_DP_FORCE_SCHEDULE")
    os.environ["MIST_DP_FORCE_SCHEDULE"] = schedule
    try:
        rc = lib.mist_dp_run_sized(sp, ctypes.byref(costs), d_t.data_ptr(), d_g.data_ptr(), n, mode, out[0].data_ptr(),
                                   out[1].data_ptr(), out[2].data_ptr(), argmin.data_ptr() if want_path else None,
                                   path.data_ptr() if want_path else None, scratch.data_ptr(), floats, stream)
    finally:
        if old is None:
            del os.environ["MIST_DP_FORCE_SCHEDULE"]
        else:
            os.environ["MIST_DP_FORCE_SCHEDULE"] = old
    _lib.check(rc, schedule)
    torch.cuda.synchronize()
    out = out.cpu().numpy().view(np.int32)
    return (out, path.cpu().numpy()) if want_path else out


@pytest.mark.parametrize(
    "L,D,meshes,S,n,quantum,rule",
    [
        (1, 1, [(1, 1)], 1, 3, None, 0),                                                     # one state
        (1, 4, [(1, 2), (1, 4)], 1, 3, None, 0),
        (5, 1, [(1, 1)], 2, 3, None, 0),                                                     # more stages than devices
        (9, 8, [(1, 1), (1, 2), (1, 4), (2, 4)], 9, 600, 0.125, 0),                          # more instances than workgroups
        (16, 64, [(1, 1), (1, 8), (2, 8), (4, 8), (8, 8)], 8, 40, 0.0625, 1),                # D a multiple of 64
        (33, 65, [(1, 1), (1, 5), (5, 5), (5, 13)], 12, 40, 0.0625, 2),                      # and one above
        (66, 33, [(1, k) for k in range(1, 17)], 9, 30, 0.03125, 0),                         # rows above 64, the most meshes
        (48, 128, [(1, 1), (1, 2), (1, 8), (2, 8), (16, 8)], 16, 30, 0.03125, 0),
        (80, 256, [(1, 4), (1, 8), (2, 8), (4, 8), (8, 8), (16, 8), (32, 8)], 16, 24, 0.03125, 0),
    ],
)
@pytest.mark.parametrize("mode", [0, 1], ids=["threshold", "bottleneck"])
def test_history_schedule_gives_what_the_step_schedule_gives(L, D, meshes, S, n, quantum, rule, mode):
    rng = np.random.default_rng(L * 1000 + D + mode)
    tabs = [_random_tables(rng, len(meshes), S, L, quantum=quantum) for _ in range(3)]
    tmax = rng.uniform(0.05, 1.1, size=n).astype(np.float32)
    g_index = rng.integers(0, 3, size=n).astype(np.int32)
    args = (meshes, L, D, S, S, rule, tabs, g_index, tmax, mode)
    want, got = _run(*args, "step"), _run(*args, "history")
    feasible = want[0] >= 0
    assert feasible.any() or L * D <= 5
    assert np.array_equal(want[0], got[0])
    assert np.array_equal(want[1], got[1])
    assert np.array_equal(want[2][feasible], got[2][feasible])
    # the partitions: the other schedule's back-pointers, walked
    with_path, path = _run(*args, "history", want_path=True)
    assert np.array_equal(with_path, got)
    assert np.array_equal(path, _run(*args, "step", want_path=True)[1])
    # empty slots of a batch are infeasible and leave the others as they are
    g_index[::2] = -1
    again = _run(meshes, L, D, S, S, rule, tabs, g_index, tmax, mode, "history")
    assert (again[0][::2] == -1).all()
    assert np.array_equal(again[:, 1::2], got[:, 1::2])


@pytest.mark.parametrize("L,S,n,quantum", [(1, 1, 3, None), (9, 9, 40, 0.125), (37, 16, 30, 0.0625), (64, 3, 9, 0.0625),
                                           (65, 32, 70, 0.03125), (100, 8, 20, 0.03125)])
@pytest.mark.parametrize("rule", [0, 1, 2])
@pytest.mark.parametrize("mode", [0, 1], ids=["threshold", "bottleneck"])
def test_one_mesh_schedule_gives_what_the_step_schedule_gives(L, S, n, quantum, rule, mode):
    rng = np.random.default_rng(L * 1000 + rule + mode)
    tabs = [_random_tables(rng, 1, S, L, quantum=quantum) for _ in range(3)]
    tmax = rng.uniform(0.05, 1.1, size=n).astype(np.float32)
    g_index = rng.integers(0, 3, size=n).astype(np.int32)
    g_index[-1] = -1
    args = ([(2, 4)], L, 0, S, S, rule, tabs, g_index, tmax, mode)
    want, want_path = _run(*args, "step", free=True, want_path=True)
    want = want[:, :-1]
    got, path = _run(*args, "", free=True, want_path=True)
    assert np.array_equal(got, _run(*args, "", free=True))
    assert np.array_equal(path[:-1], want_path[:-1])
    assert (path[-1] == -1).all()
    feasible = want[0] >= 0
    assert got[0, -1] == -1
    got = got[:, :-1]
    assert np.array_equal(want[0], got[0])
    assert np.array_equal(want[1], got[1])
    assert np.array_equal(want[2][feasible], got[2][feasible])


@pytest.mark.parametrize("L, D, S", [(40, 5, 8), (40, 11, 12), (40, 4, 8), (40, 10, 12), (7, 5, 7), (70, 17, 16)])
@pytest.mark.parametrize("mode", [0, 1], ids=["threshold", "bottleneck"])
def test_instances_whose_states_run_out(L, D, S, mode):
    """Stages take two devices each: with the third, sixth or ninth stage count no state is left, behind an
    answer (D even) or without one, while further instances wait for the same workgroups."""
    rng = np.random.default_rng(L + D + mode)
    meshes, n = [(1, 2), (2, 1)], 600
    tabs = [_random_tables(rng, len(meshes), S, L, quantum=0.0625) for _ in range(2)]
    tmax = rng.choice([0.0, 0.5, 2.0], size=n).astype(np.float32)
    g_index = rng.integers(-1, 2, size=n).astype(np.int32)
    args = (meshes, L, D, S, S, 0, tabs, g_index, tmax, mode)
    want = _run(meshes, L, D, S, S, 0, tabs, np.maximum(g_index, 0), tmax, mode, "step")
    feasible = (want[0] >= 0) & (g_index >= 0)
    assert feasible.any() == (D % 2 == 0)
    got, path = _run(*args, "history", want_path=True)
    assert np.array_equal(got[0], np.where(g_index >= 0, want[0], -1))
    assert np.array_equal(got[1:, feasible], want[1:, feasible])
    assert ((path[:, 0, 0] >= 0) == feasible).all()
    assert np.array_equal(got, _run(*args, "history"))
