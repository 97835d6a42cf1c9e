"""Search with DP instances that end early, and on multiples of the meshes' common divisor, against the
reference's scan."""
import numpy as np
import pytest

from tests.test_gpu_inter import _synthetic_results

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed, L, D, meshes, quantum, inf_frac, structured", [
    (0, 9, 8, [(1, 1), (1, 2), (1, 4), (1, 8)], 1 / 16, 0.2, True),
    (1, 12, 16, [(1, 4), (1, 8), (2, 8)], 1 / 64, 0.1, True),    # multiples of four devices
    (2, 12, 24, [(1, 6), (1, 12), (2, 12)], 1 / 64, 0.3, False),  # of six
    (3, 24, 32, [(1, 1), (1, 2), (1, 4), (1, 8), (2, 8), (4, 8)], 1 / 512, 0.1, True),
    (4, 10, 80, [(1, 1), (1, 8), (2, 8), (5, 8)], 1 / 128, 0.1, True),   # 80 columns, or 10
    (5, 7, 12, [(1, 5), (1, 7)], 1 / 16, 0.0, False),             # divisor 1 of D and the meshes
    (6, 8, 16, [(1, 4), (2, 4)], 1 / 16, 1.0, True),              # no stage anywhere
])
def test_search_equals_the_reference_scan(monkeypatch, seed, L, D, meshes, quantum, inf_frac, structured):
    from mist_amd import inter_tuning
    from oracle import inter_dp
    from oracle.dp_c import dp_impl_c

    rng = np.random.default_rng(400 + seed)
    Gs, S, slot = [1, 4, 16], 1, 0
    ours, theirs = _synthetic_results(rng, 2, Gs, meshes, L, min(D, L), S, quantum, inf_frac, structured)
    want = [inter_dp.inter_stage_tune(L, D, meshes, Gs, r, slot, dp=dp_impl_c) for r in theirs]
    assert inf_frac == 1.0 or any(sol is not None for _, sol in want)
    for rates in ("1", "0"):
        monkeypatch.setenv("MIST_DP_RATES", rates)
        assert inter_tuning.inter_stage_tune_batch(L, D, meshes, Gs, ours, slot=slot) == want, rates
