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


def _tune(samples, exhaustive=False):
    from mist_amd.config import tp_candidates
    from mist_amd.intra_tuning import IntraStageTuner

    cfg, tables = tiny_plan(2, layers=13, hardware__num_nodes=2, hardware__num_gpus_per_node=4,
                            training__global_batch_size=48, hardware__memory_capacity=9.0)
    tuner = IntraStageTuner(tables, 13, [(1, 1), (1, 4), (2, 4)], [3, 6, 24], tp_candidates(cfg)[0], cfg,
                            sample_size=samples, exhaustive=exhaustive)
    return tuner, tuner.tune().device


def _same(got, want):
    import torch

    return all(torch.equal(getattr(got, kind)[v], getattr(want, kind)[v])
               for v in range(4) for kind in ("index", "stable", "delta"))


# (a chunk takes 512.5 doubles, and one more)
@pytest.mark.parametrize("samples, extra", [(1, 0), (1, 512), (1, 513), (1, 4000), (1, 4104), (30, 0), (30, 100001)])
def test_workspace_with_room_for_a_shorter_log(monkeypatch, samples, extra):
    from mist_amd import _lib, intra_tuning

    _, want = _tune(samples, exhaustive=True)
    free = 1 << 36
    monkeypatch.setattr(intra_tuning, "_free_device_bytes", lambda device: free)
    monkeypatch.setattr(intra_tuning, "ROW_TERMS_LEAST_BYTES", 0)  # (every plan asks)
    monkeypatch.setattr(intra_tuning, "LOG_FREE_SHARE", 8 * extra / free)
    tuner, got = _tune(samples)
    problem = tuner._plan["problem"]
    least = _lib.load().mist_reduce_workspace_least_doubles(
        *(int(problem[key][0]) for key in ("reduce_cells", "reduce_supers", "reduce_items")), samples)
    assert tuner._dev_plan["partial_cost"].numel() == int(problem["reduce_doubles"][0]) == least + extra
    assert _same(got, want)
    # one double short of what the launches need without a log
    problem["reduce_doubles"] = least - 1
    with pytest.raises(_lib.MistLibraryError, match="reduce workspace"):
        tuner.run_prepared(tuner._plan, tuner._dev_plan)


def test_workspace_where_memory_is_short(monkeypatch):
    """An allocation that fails with the log is tried without it; one that fails without it fails."""
    import torch

    from mist_amd import _lib

    _, want = _tune(3, exhaustive=True)
    lib, empty, asked = _lib.load(), torch.empty, []
    whole, least = ({}, {})

    def sizes_of(kind, function):
        def sizes(*args):
            kind["doubles"] = function(*args)
            return kind["doubles"]
        return sizes

    monkeypatch.setattr(lib, "mist_reduce_workspace_doubles", sizes_of(whole, lib.mist_reduce_workspace_doubles))
    monkeypatch.setattr(lib, "mist_reduce_workspace_least_doubles",
                        sizes_of(least, lib.mist_reduce_workspace_least_doubles))

    def short(refused):
        def allocate(size, *args, **kwargs):
            asked.append(size)
            if size in refused():
                raise torch.cuda.OutOfMemoryError("short of memory")
            return empty(size, *args, **kwargs)
        return allocate

    monkeypatch.setattr(torch, "empty", short(lambda: [whole.get("doubles")]))
    tuner, got = _tune(3)
    assert whole["doubles"] in asked and tuner._dev_plan["partial_cost"].numel() == least["doubles"]
    assert _same(got, want)
    monkeypatch.setattr(torch, "empty", short(lambda: [whole.get("doubles"), least.get("doubles")]))
    with pytest.raises(torch.cuda.OutOfMemoryError):
        _tune(3)


@pytest.mark.parametrize("where", ["tables", "costs", "library", "elsewhere"])
def test_search_where_memory_is_short_beside_the_log(monkeypatch, where):
    """Tables, cost tables or the library's own buffers that find no memory beside the log: the search goes on
    without it.  A second failure, and any other error, is the caller's."""
    import torch

    from mist_amd import _lib
    from mist_amd.tune_one_case import PreparedSearch

    cfg, _ = tiny_plan(2, layers=13, hardware__num_nodes=2, hardware__num_gpus_per_node=4, training__global_batch_size=48)
    search = PreparedSearch(cfg)
    want = search.run()
    problem, empty, failures = search.plan["problem"], torch.empty, []
    assert int(problem["reduce_doubles"][0]) > search.plan["reduce_least"]
    total = search.tuner._table_layout()[1][-1]
    lib = _lib.load()
    bounded = lib.mist_inter_stage_search_bounded
    size = {"tables": 2 * total, "costs": 2 * total // search.tuner.table_samples}.get(where)
    dtype = torch.float64 if where == "tables" else torch.float32

    def allocate(shape, *args, **kwargs):
        n = shape[0] if isinstance(shape, tuple) else shape
        if n == size and kwargs.get("dtype") is dtype and most > len(failures):
            failures.append(n)
            raise torch.cuda.OutOfMemoryError("HIP out of memory")
        return empty(shape, *args, **kwargs)

    def searched(*args):
        if where not in ("library", "elsewhere") or len(failures) >= most:
            return bounded(*args)
        failures.append(where)
        raise _lib.MistLibraryError("hipMalloc failed: out of memory" if where == "library" else "null pointer argument")

    monkeypatch.setattr(torch, "empty", allocate)
    monkeypatch.setattr(lib, "mist_inter_stage_search_bounded", searched)
    most = 1
    if where == "elsewhere":
        with pytest.raises(_lib.MistLibraryError, match="null pointer"):
            search.run()
        assert int(problem["reduce_doubles"][0]) > search.plan["reduce_least"]
        return
    assert search.run() == want and len(failures) == 1
    assert search.dev_plan["partial_cost"].numel() == int(problem["reduce_doubles"][0]) == search.plan["reduce_least"]
    assert search.dev_plan["partial_cost"] is search.dev_plan["workspaces"][0]["partial_cost"]
    assert search.run() == want
    most = 2
    with pytest.raises((torch.cuda.OutOfMemoryError, _lib.MistLibraryError), match="out of memory"):
        search.run()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert search.run() == want
