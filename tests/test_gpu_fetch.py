"""``mist_fetch_tables`` at the sizes where its chunks of 1 MiB and their pieces begin and end, against copies and
the host's decoding of the strategy rows."""
import ctypes

import numpy as np
import pytest
import yaml

from tests.util import CONFIG_DIR

pytestmark = pytest.mark.gpu

PER_CHUNK = (1 << 20) // 80  # strategy rows


@pytest.mark.parametrize("sizes", [
    [("rows", 1)], [("rows", PER_CHUNK)], [("rows", PER_CHUNK + 1)], [("rows", 7 * PER_CHUNK - 3)],
    [("doubles", 1)], [("doubles", 131072)], [("doubles", 131073)], [("doubles", 1000003)],
    [("doubles", 3), ("rows", 5), ("doubles", 0), ("none", 4), ("rows", 40001), ("doubles", 131071), ("none", 20000)],
    [("doubles", 1 + i % 3) for i in range(50)] + [("rows", 0)],
])
def test_tables_and_rows_on_the_host(sizes):
    import torch

    from mist_amd import _lib
    from mist_amd.config import MistConfig
    from mist_amd.intra_tuning import IntraStageTuner
    from mist_amd.layer_tables import LayerTables

    with open(f"{CONFIG_DIR}/gpt-7b-b512-4x8.yaml") as f:
        cfg = MistConfig(yaml.safe_load(f))
    tuner = IntraStageTuner(LayerTables(cfg), 32, [(1, 1), (2, 8)], [8], 2, cfg, sample_size=1)
    plan = tuner.prepare()
    group = len(plan["groups"]) - 1
    assert group >= 0
    record = plan["groups"][group]
    space = plan["spaces"][0, int(record["g_index"]), int(record["q_index"])]
    rng = np.random.default_rng(len(sizes))
    lib = _lib.load()
    with torch.cuda.device(tuner.device):
        groups = tuner.upload(plan)["groups"]
        items, kept, got, want = (_lib.FetchItem * len(sizes))(), [], [], []
        for i, (kind, n) in enumerate(sizes):
            if kind == "doubles":
                source = torch.from_numpy(rng.normal(size=n)).cuda()
                want.append(source.cpu().numpy())
            else:
                index = rng.integers(-1, space.n_rows, size=n).astype(np.int32)
                index[:1], index[-1:] = 0, space.n_rows - 1
                source = torch.from_numpy(index).cuda()
                want.append(space.decode(index) if kind == "rows" else np.full((n, 10), np.inf))
            kept.append(source if n else torch.zeros(1, device="cuda", dtype=source.dtype))
            got.append(np.full(want[-1].shape if n else (1,), 7.0))
            items[i] = _lib.FetchItem(kept[-1].data_ptr(), got[-1].ctypes.data, n, kind != "doubles",
                                      -1 if kind == "none" else group)
        for _ in range(2):
            _lib.check(lib.mist_fetch_tables(items, len(sizes), groups.data_ptr(), group + 1, None), "mist_fetch_tables")
    for (kind, n), a, b in zip(sizes, got, want):
        assert np.array_equal(a, b if n else [7.0]), (kind, n)
