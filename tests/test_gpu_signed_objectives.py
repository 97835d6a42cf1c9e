"""Minima of objectives of either sign against the CPU oracle.

``r stable + delta / G`` is negative where the first micro-batch is cheaper than the later ones
(they swap weights in) by more than ``r`` times the rest: small alpha samples, few accumulation
steps.  Small plans whose tables hold such cells, as the oracle finds them.
"""
import numpy as np
import pytest

from mist_amd.config import MistConfig
from mist_amd.configs.make_configs import PLANS, build, ratios
from mist_amd.layer_tables import LayerTables
from tests.util import assert_same_f64

pytestmark = pytest.mark.gpu


def _plan(seed, base, layers, mesh, batch, capacity, step=0.25, batch_sizes=None, vocab=None, disable_tp=False, **tuning):
    plan = dict(PLANS[base - 1], batch=batch, nodes=mesh[0], gpus=mesh[1], off=ratios(step), mem=capacity)
    plan["model"] = dict(plan["model"], num_hidden_layers=layers)
    if batch_sizes:
        plan["b_cands"] = batch_sizes
    if vocab:
        plan["model"]["vocab_size"] = vocab
    raw = build(seed, plan)
    raw["tuning"].update(tuning)
    raw["disable_tp_tuning"] = disable_tp
    cfg = MistConfig(raw)
    return cfg, LayerTables(cfg)


def _oracle(cfg, tables, mesh, G, tp, samples):
    """(index, stable, delta) of the four tables, and how many of their minima are negative."""
    from oracle.pareto import alpha_ratios
    from oracle.stage import batched_tune_best_latency_for_stage

    L = cfg.model.num_hidden_layers
    n_p = min(mesh[0] * mesh[1], L, G)
    found = batched_tune_best_latency_for_stage(
        tables, cfg, list(range(n_p)), list(range(1, L + 1)), list(range(L + 1)), *mesh, G, tp_size=tp,
        sample_size=samples, inner="c")
    negative = []
    for v, (stable, delta, _, index) in enumerate(found):
        share = (delta.astype(np.float32) / np.float32(G)).astype(np.float64) if v == 0 else delta / G
        with np.errstate(invalid="ignore"):
            negative.append(int(((alpha_ratios(samples) * stable + share < 0) & (index >= 0)).sum()))
    return [(index, stable, delta) for stable, delta, _, index in found], negative


def _hold(got, want, slots):
    for v, suffix in enumerate(("", "_with_pre", "_with_post", "_no_pp")):
        index, stable, delta = (a[..., slots] for a in want[v])
        mine = getattr(got, "indices" + suffix)[0, 0][..., slots]
        assert np.array_equal(mine, index), f"indices{suffix}: {int((mine != index).sum())} of {index.size} differ"
        assert_same_f64(got.costs_f64("stable", v)[0, 0][..., slots], stable, "stable" + suffix)
        assert_same_f64(got.costs_f64("delta", v)[0, 0][..., slots], delta, "delta" + suffix)


# seed, model, layers, mesh, G, samples, batch, capacity in GB
SIGNED = [
    (1035, 2, 6, (1, 4), 2, 10, 8, 18.0),
    (299, 2, 8, (1, 4), 2, 20, 32, 32.0),
    (144, 2, 4, (1, 8), 2, 30, 16, 8.0),
    (257, 2, 7, (1, 2), 4, 30, 32, 28.0),
    (365, 3, 6, (1, 4), 4, 30, 16, 24.0),
]


@pytest.mark.parametrize("exhaustive, seeded", [(False, True), (False, False), (True, False)],
                         ids=["seeded", "empty-minima", "every-cell"])
@pytest.mark.parametrize("seed, base, layers, mesh, G, samples, batch, capacity", SIGNED)
def test_tables_with_negative_minima(seed, base, layers, mesh, G, samples, batch, capacity, exhaustive, seeded,
                                     monkeypatch):
    """All samples together, and the first one (the smallest ratio) alone through the one-sample
    kernels, as the uniform search asks for it."""
    from mist_amd import intra_tuning
    from mist_amd.intra_tuning import IntraStageTuner

    if not seeded:
        monkeypatch.setattr(intra_tuning, "SCOUT_MIN_STAGES", 0)
    cfg, tables = _plan(seed, base, layers, mesh, batch, capacity)
    want, negative = _oracle(cfg, tables, mesh, G, 1, samples)
    assert all(n > 0 for n in negative), negative
    for slots in (list(range(samples)), [0]):
        got = IntraStageTuner(tables, layers, [mesh], [G], 1, cfg, sample_size=samples, sample_slots=slots,
                              exhaustive=exhaustive).tune()
        _hold(got, want, slots)


@pytest.mark.parametrize("seed, base, layers, gpus, batch, batch_size, capacity, disable_tp, granularity", [
    (477, 3, 2, 4, 8, 1, 12.0, True, "uniform-pp"),
    (750, 3, 5, 2, 4, 1, 30.0, False, "uniform-pp"),
    (787, 3, 5, 4, 8, 1, 30.0, True, "uniform-pp"),
    (2372, 3, 5, 2, 2, 1, 30.0, False, "uniform-device-pp-mip"),
])
def test_tune_whose_answer_has_a_negative_objective(seed, base, layers, gpus, batch, batch_size, capacity, disable_tp,
                                                    granularity):
    from mist_amd.tune_one_case import tune
    from oracle.tune import tune as oracle_tune

    cfg, tables = _plan(seed, base, layers, (1, gpus), batch, capacity, step=0.5, batch_sizes=[batch_size],
                        disable_tp=disable_tp, tuning_granularity=granularity, sample_size=30)
    want = oracle_tune(cfg, tables)
    assert want[1] is not None
    assert tune(cfg) == want


@pytest.mark.parametrize("exhaustive", [False, True], ids=["pruned", "every-cell"])
@pytest.mark.parametrize("seed, layers, capacity, vocab", [(601, 8, 33.9, 622444), (2027, 7, 36.4, 774180)])
def test_minima_far_smaller_than_their_operands(seed, layers, capacity, vocab, exhaustive):
    """G = 3: the base objective rounds ``delta / G`` to float32.  Where it nearly cancels
    ``r stable``, that rounding is more than a millionth of the minimum: a winner whose exact sum
    lies above the minimum by more than such a share of it must not be pruned.  (Picked so that no
    first-stage minimum keeps those cells open.)"""
    from mist_amd.intra_tuning import IntraStageTuner
    from oracle.pareto import alpha_ratios

    mesh, G, samples, batch = (1, 2), 3, 30, 12
    cfg, tables = _plan(seed, 2, layers, mesh, batch, capacity, vocab=vocab)
    want, negative = _oracle(cfg, tables, mesh, G, 1, samples)
    (index, stable, delta), pre_index = want[0], want[1][0]
    ratio = alpha_ratios(samples)
    with np.errstate(invalid="ignore"):
        cost = ratio * stable + (delta.astype(np.float32) / np.float32(G)).astype(np.float64)
        cancels = (index >= 0) & (pre_index < 0) & (ratio * stable + delta / G > cost + 1e-6 * np.abs(cost))
    assert cancels.any() and negative[0] > 0
    got = IntraStageTuner(tables, layers, [mesh], [G], 1, cfg, sample_size=samples, exhaustive=exhaustive).tune()
    _hold(got, want, list(range(samples)))


@pytest.mark.parametrize("seed, base, layers, mesh, G, batch, capacity", [
    (326, 2, 7, (1, 4), 3, 24, 28.0), (299, 3, 8, (1, 2), 3, 12, 48.0), (318, 2, 7, (1, 4), 7, 28, 42.0),
])
def test_stage_operator_with_a_count_that_is_no_power_of_two(seed, base, layers, mesh, G, batch, capacity):
    from mist_amd.batched_module_analyzer import batched_tune_best_latency_for_stage as on_gpu
    from oracle.stage import batched_tune_best_latency_for_stage as on_cpu

    cfg, tables = _plan(seed, base, layers, mesh, batch, capacity)
    shape = (range(2), range(1, layers + 1), range(layers + 1), *mesh, G)
    for samples in (1, 30):
        got = on_gpu(tables, None, None, *shape, cfg, tp_size=1, sample_size=samples)
        want = on_cpu(tables, cfg, *map(list, shape[:3]), *mesh, G, tp_size=1, sample_size=samples, inner="c")
        for v in range(4):
            for i in range(3):
                assert_same_f64(got[v][i], want[v][i], f"{samples} samples, result {i} of table {v}")
