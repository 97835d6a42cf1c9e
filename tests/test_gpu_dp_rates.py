"""Search with DP instances that end early, and on multiples of the meshes' common divisor, against the
reference's scan; costs of either sign."""
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


def _negate(rng, ours, theirs, negated, zeros):
    """A share of the costs negated on all meshes but the last, a share of the last mesh's -0.0, in both."""
    import torch

    whole, n_g = ours[0].batch, len(theirs[0].costs_stable)
    for v, name in enumerate(("", "_with_pre", "_with_post", "_no_pp")):
        cells = {"costs_stable": whole.stable[v].cpu().numpy(), "costs_delta": whole.delta[v].cpu().numpy()}
        held = np.isfinite(cells["costs_stable"])
        flip, zero = (rng.random(held.shape) < negated) & held, (rng.random(held.shape) < zeros) & held
        flip[:, -1], zero[:, :-1] = False, False
        for name_of, device in (("costs_stable", whole.stable[v]), ("costs_delta", whole.delta[v])):
            cells[name_of][flip] *= -1.0
            cells[name_of][zero] = -0.0
            device.copy_(torch.from_numpy(cells[name_of]))
            for t, r in enumerate(theirs):
                getattr(r, name_of + name)[...] = cells[name_of][t * n_g:(t + 1) * n_g]


@pytest.mark.parametrize("negated, zeros", [(0.1, 0.0), (0.1, 0.3), (0.002, 0.02), (0.0, 0.3)])
@pytest.mark.parametrize("L, D, meshes", [
    (9, 8, [(1, 1), (1, 2), (1, 4), (1, 8)]),
    (12, 16, [(1, 4), (1, 8), (2, 8)]),
    (16, 32, [(1, 1), (1, 2), (1, 8), (4, 8)]),
    (17, 64, [(1, 8), (2, 8), (8, 8)]),  # where the rates are used by themselves
])
def test_costs_of_either_sign(monkeypatch, L, D, meshes, negated, zeros):
    """The end of an instance is proved for costs that are not negative: zeros of either sign do not hide those
    that are, and the smallest cost of a mesh is that of all shares of its stage counts."""
    from mist_amd import inter_tuning
    from oracle import inter_dp
    from oracle.dp_c import dp_impl_c

    rng = np.random.default_rng(L)
    Gs = [1, 4, 16]
    ours, theirs = _synthetic_results(rng, 2, Gs, meshes, L, min(D, L), 1, 1 / 64, 0.2, structured=True)
    _negate(rng, ours, theirs, negated, zeros)
    want = [inter_dp.inter_stage_tune(L, D, meshes, Gs, r, 0, dp=dp_impl_c) for r in theirs]
    assert any(cost < 0 for cost, _ in want) or negated < 0.01
    for rates in ("1", "0", ""):
        monkeypatch.setenv("MIST_DP_RATES", rates)
        assert inter_tuning.inter_stage_tune_batch(L, D, meshes, Gs, ours) == want, rates
