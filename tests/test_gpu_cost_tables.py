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


@pytest.mark.parametrize("L, P1, Gn, samples", [
    (3, 2, 33001, 1), (20, 2, 2003, 1), (62, 2, 301, 1), (254, 2, 13, 1),  # four cells a lane: 3, 6, 8, 6 sets
    (3, 2, 12007, 2), (20, 2, 305, 2), (63, 2, 51, 2), (300, 1, 7, 1),  # a cell a lane: 4, 3, 5, 8
])
def test_several_sets_of_rows_a_workgroup(L, P1, Gn, samples):
    """Tables of so many rows that a workgroup takes 3 to 8 sets of them in turn, of short rows and long ones:
    accumulation counts that change between the sets and, where one has few rows, several times inside one."""
    import ctypes

    import torch

    from mist_amd import _lib
    from mist_amd.intra_tuning import DeviceTables

    rng = np.random.default_rng(L + samples)
    Q, slot = 3, samples - 1
    shapes = [(Gn, Q, P1, L, L + 1, samples)] * 2 + [(Gn, Q, L, L + 1, samples), (Gn, Q, L + 1, samples)]
    grad_accum = rng.integers(1, 50, size=Gn).astype(np.int32)
    stable, delta, index = [], [], []
    for shape in shapes:
        s, d = (rng.integers(1, 4096, size=shape, dtype=np.int16).astype(np.float64) / 256 for _ in range(2))
        none = rng.integers(0, 2, size=shape, dtype=np.int8) == 0
        s[none] = d[none] = np.inf
        stable.append(s), delta.append(d), index.append(np.where(none, -1, 7).astype(np.int32))
    tables = DeviceTables(*[[torch.from_numpy(a).cuda() for a in kind] for kind in (stable, delta, index)])
    got = [[torch.full(shape[:-1], -9.0, dtype=torch.float32, device="cuda") for shape in shapes] for _ in range(2)]
    problem = np.zeros(1, dtype=_lib.PROBLEM_DTYPE)
    problem["num_layers"], problem["p_dim"], problem["sample_size"] = L, P1, samples
    problem["num_grad_accum"], problem["num_mesh"] = Gn, Q
    d_G, tabs = torch.from_numpy(grad_accum).cuda(), tables.as_struct()
    pointers = [(ctypes.c_void_p * 4)(*[t.data_ptr() for t in kind]) for kind in got]
    _lib.check(_lib.load().mist_dp_cost_tables(
        ctypes.c_void_p(problem.ctypes.data), ctypes.byref(tabs), d_G.data_ptr(), slot, *pointers,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "mist_dp_cost_tables")
    for v, shape in enumerate(shapes):
        G = grad_accum.astype(np.float32).reshape((-1,) + (1,) * (len(shape) - 2))
        want = stable[v][..., slot].astype(np.float32) + delta[v][..., slot].astype(np.float32) / G
        want_min = np.minimum.accumulate(want, axis=-1)
        for mine, theirs in zip((got[0][v], got[1][v]), (want, want_min)):
            assert np.array_equal(mine.cpu().numpy().view(np.int32), theirs.view(np.int32)), v
