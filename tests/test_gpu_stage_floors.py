"""Stage summaries from the key terms, with the parts that rows share evaluated once, against those of rows that
evaluate everything: every byte, for lists of ratios whose blocks are shorter, as long as and longer than a stage."""
import ctypes

import numpy as np
import pytest
import yaml

from tests.util import CONFIG_DIR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("runs", ["0", "1"])
@pytest.mark.parametrize("n_dense, n_sparse, far", [
    (1, 1, False), (2, 1, False), (1, 2, False), (3, 2, False), (4, 4, False), (5, 3, False), (6, 5, False), (7, 11, False),
    (13, 4, False), (1, 32, False), (32, 2, False), (1, 1, True), (5, 2, True),
])
def test_summaries_from_keys_equal_those_of_the_rows(monkeypatch, n_dense, n_sparse, far, runs):
    import torch

    from mist_amd import _lib
    from mist_amd.config import MistConfig
    from mist_amd.intra_tuning import IntraStageTuner
    from mist_amd.layer_tables import LayerTables

    monkeypatch.setenv("MIST_STAGE_FLOOR_RUNS", runs)
    with open(f"{CONFIG_DIR}/gpt-1.3b-b8-1x2.yaml") as f:
        raw = yaml.safe_load(f)
    raw["hardware"].update(num_nodes=2, num_gpus_per_node=4)
    raw["training"]["global_batch_size"] = 32
    ratios = lambda n: [round(float(x), 4) for x in np.linspace(0.0, 1.0, n)]
    raw["tuning"]["search_space"].update(offloading_ratio_candidates=ratios(n_dense),
                                         sparse_offloading_ratio_candidates=ratios(n_sparse))
    cfg = MistConfig(raw)
    tuner = IntraStageTuner(LayerTables(cfg), 6, [(1, 1), (1, 4), (2, 4)], [1, 4], [1, 2], cfg, sample_size=1)
    plan = tuner.prepare()
    groups = plan["groups"]
    assert len(groups) > 0 and len(plan["batches"]) == 1
    if far:  # pairs far back in lists of 32 ratios: their blocks may have no room
        for rec in plan["batches"][0]["groups"]:
            for which in ("wo", "go"):
                n = int(rec["pair_" + which].max()) + 1
                rec[which][32 - n:] = rec[which][:n].copy()
                rec["pair_" + which][:int(rec["n_pair"])] += 32 - n
    found = []
    with torch.cuda.device(tuner.device):
        dev = tuner.upload(plan)
        for keys in (dev["key_terms"].data_ptr(), None):
            dev["stage_floor"].fill_(-7.0)
            _lib.check(_lib.load().mist_row_terms(
                ctypes.c_void_p(plan["problem"].ctypes.data), dev["groups"].data_ptr(), dev["n_groups"],
                dev["terms_prefix"].data_ptr(), dev["n_terms_blocks"], dev["row_terms"].data_ptr(),
                dev["stage_floor"].data_ptr(), keys, None), "mist_row_terms")
            torch.cuda.synchronize()
            found.append(dev["stage_floor"].cpu().numpy().reshape(-1, 32)[:, :_lib.TERM_NAMES.index("gcb") + 5])
    n_stages = int((-(-groups["n_rows"] // _lib.STAGE_ROWS)).sum())
    assert int((found[0][:, 0] != -7.0).sum()) == n_stages
    assert np.array_equal(found[0], found[1])
