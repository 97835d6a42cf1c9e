"""The calls a user of this framework makes, at the sizes they are made with.

A user has a model, a cluster and a batch size and wants the best parallelisation strategy: one
``tune`` of a configuration object, with one of the tuning granularities.  The clusters go from
two GPUs to 32 nodes of eight, the models from 1.3 to 70 billion parameters; the configuration
object is what the program has in hand, every call builds its search from it.  Beside ``tune``
stand the two calls that a program which keeps its own inter-stage search makes (the tables of
``intra_stage_tune`` for one tensor-parallel size, ``batched_tune_best_latency_for_stage`` for one
mesh and accumulation count) and ``analyze``, which prices one given strategy.

Shapes are those of ``mist_amd/configs``; the link, copy and interference coefficients and the
operator efficiencies of a case are drawn from its seed with the generator of those plans.
"""
import math

import numpy as np

from mist_amd.analysis import analyze
from mist_amd.batched_module_analyzer import batched_tune_best_latency_for_stage
from mist_amd.config import MistConfig, tp_candidates
from mist_amd.configs.make_configs import PLANS, build, ratios
from mist_amd.intra_tuning import intra_stage_tune
from mist_amd.layer_tables import LayerTables
from mist_amd.search_space import (SearchSpaceFactory, _get_device_mesh_candidates,
                                   _get_grad_accumu_steps_candidates)
from mist_amd.tune_one_case import tune

#: Model shapes with the memory, peak and bandwidth of the GPUs they are planned for.  ``7b-l4`` is
#: the plan of tests/golden/tuned_configs on 24 GB cards; the others are mist_amd/configs.
FAMILIES = {name: dict(PLANS[i]) for i, name in enumerate(("1.3b", "7b", "13b", "22b", "70b"))}
FAMILIES["7b-l4"] = dict(
    file="llama-7b", seq=2048, dtype="float16", mem=24.0, peak=121.0, hbm=300.0, b_cands=[1, 2, 4],
    model=dict(name="llama-7b", hidden_size=4096, num_attention_heads=32, vocab_size=50304, use_flash_attn=True,
               intermediate_size=11008, mlp_type="gated_mlp", normalization="rmsnorm",
               position_embedding_type="rotary"),
)
#: Largest drawn values of a family: layers, nodes, batch size, and parameters per layer in billions.
LIMITS = {"1.3b": (24, 1, 64, 0.054), "7b-l4": (32, 2, 256, 0.21), "7b": (32, 4, 512, 0.21),
          "13b": (40, 8, 1024, 0.32), "22b": (48, 16, 1536, 0.46), "70b": (80, 32, 2048, 0.86)}

#: ``step``: spacing of the offload ratios, 0 for the search space the tuner takes without a
#: ``search_space`` block.
TUNE = dict(kind="tune", granularity="inter-stage", samples=1, step=0.1, ckpt_tuning=True)


def listed():
    mip = dict(granularity="uniform-device-pp-mip", samples=30)
    return [
        # the smallest call: what a given four-stage strategy costs in time and memory
        dict(name="analyze-7b-4-stages", kind="analyze", family="7b", layers=32, batch=512, nodes=4, gpus=8,
             stages=4, grad_accum=16),
        # a workstation: two GPUs, small batch, coarse ratios; launches and host work count
        dict(TUNE, name="tune-1.3b-1x2", family="1.3b", layers=24, batch=8, nodes=1, gpus=2, step=0.25),
        # one node of small cards with the default granularity and the default search space
        dict(TUNE, name="tune-7b-1x8-mip", family="7b-l4", layers=32, batch=128, nodes=1, gpus=8, **dict(mip, step=0)),
        # the headline plan, with each way of dividing the pipeline that users choose from
        dict(TUNE, name="tune-7b-4x8", family="7b", layers=32, batch=512, nodes=4, gpus=8),
        dict(TUNE, name="tune-7b-4x8-mip", family="7b", layers=32, batch=512, nodes=4, gpus=8, **mip),
        dict(TUNE, name="tune-7b-2x8-uniform", family="7b", layers=32, batch=256, nodes=2, gpus=8,
             granularity="uniform-pp"),
        # many micro-batch sizes; then the same family at odd sizes, one mesh for all stages, no checkpoint tuning
        dict(TUNE, name="tune-13b-8x8", family="13b", layers=40, batch=1024, nodes=8, gpus=8),
        dict(TUNE, name="tune-13b-4x8-device", family="13b", layers=37, batch=768, nodes=4, gpus=8,
             granularity="uniform-device-pp", ckpt_tuning=False),
        # the two largest searches: the finest ratios, and the largest cluster and deepest model
        dict(TUNE, name="tune-22b-16x8", family="22b", layers=48, batch=1536, nodes=16, gpus=8, step=0.05),
        dict(TUNE, name="tune-70b-32x8", family="70b", layers=80, batch=2048, nodes=32, gpus=8),
        # whole tables with the default number of samples, for a program with its own search over them
        dict(name="tables-7b-tp2", kind="tables", family="7b", layers=32, batch=512, nodes=4, gpus=8, tp=2,
             samples=30, step=0.1, ckpt_tuning=True),
        # one mesh and accumulation count through the operator boundary: host arrays come back
        dict(name="stage-7b-2x8", kind="stage", family="7b", layers=32, batch=512, nodes=2, gpus=8, tp=4,
             grad_accum=32, samples=1, step=0.1, ckpt_tuning=True),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _cluster(rng, family, granularity):
    """Layers and nodes under the family's limits, with nodes enough to hold the states of the
    model (18 bytes a parameter, half of the memory), and a batch the nodes can divide.  A pipeline
    of one mesh for all stages needs a power of two of nodes."""
    max_layers, max_nodes, max_batch, params = LIMITS[family]
    if granularity == "uniform-pp":
        max_nodes, max_batch = min(max_nodes, 2), min(max_batch, 256)
    layers = _log_int(rng, min(9, max_layers), max_layers)
    gpus = rng.choice((2, 4)) if family == "1.3b" else 8
    need = max(1, math.ceil(18 * params * layers / (0.5 * FAMILIES[family]["mem"] * gpus)))
    nodes = _log_int(rng, min(need, max_nodes), max_nodes)
    if granularity in ("uniform-pp", "uniform-device-pp"):
        nodes = 1 << (nodes.bit_length() - 1)
    odd = 3 if family == "22b" or nodes % 3 == 0 else 1
    top = int(math.log2(max_batch // odd))
    low = min(top, max(3, (nodes * gpus // odd).bit_length() - 1))
    return dict(layers=layers, nodes=nodes, gpus=gpus, batch=odd << rng.randint(low, top))


def draw(rng):
    kind = rng.choices(("tune", "tables", "stage", "analyze"), (9, 1, 1, 1))[0]
    if kind == "analyze":
        layers, stages = rng.randint(9, 80), rng.choice((1, 2, 3, 4, 6, 8))
        return dict(kind=kind, family=rng.choice(("7b", "13b", "70b")), layers=layers, nodes=stages, gpus=8,
                    stages=stages, grad_accum=1 << rng.randint(1, 6), batch=0)
    if kind == "stage":
        nodes, tp = rng.choice((1, 2, 4)), rng.choice((1, 2, 4, 8))
        grad_accum = 1 << rng.randint(0, 5)
        return dict(kind=kind, family="7b", layers=rng.randint(9, 32), nodes=nodes, gpus=8, tp=tp, grad_accum=grad_accum,
                    batch=rng.choice((1, 2, 4)) * (8 * nodes // tp) * grad_accum, samples=rng.choice((1, 2, 3)), step=0.1,
                    ckpt_tuning=True)
    if kind == "tables":
        samples = _log_int(rng, 1, 30)
        return dict(_cluster(rng, "7b", "inter-stage"), kind=kind, family="7b", tp=rng.choice((1, 2, 4, 8)), samples=samples,
                    step=0.1, ckpt_tuning=True)
    family = rng.choice(tuple(LIMITS))
    granularity = rng.choices(("inter-stage", "uniform-device-pp", "uniform-device-pp-mip", "uniform-pp"), (5, 2, 3, 1))[0]
    if family in ("13b", "22b", "70b") and granularity == "uniform-pp":
        granularity = "inter-stage"
    if family in ("22b", "70b") and granularity != "inter-stage":
        granularity = rng.choice(("inter-stage", "uniform-device-pp"))
    case = dict(TUNE, family=family, granularity=granularity, ckpt_tuning=rng.random() < 0.75,
                step={"1.3b": 0.25, "7b-l4": 0, "22b": 0.05}.get(family, 0.1))
    if granularity == "uniform-device-pp-mip":
        case["samples"] = 30
    return dict(case, **_cluster(rng, family, granularity))


def _raw(case, seed):
    """The resolved configuration of a case, as a dict."""
    plan = dict(FAMILIES[case["family"]], batch=case["batch"], nodes=case["nodes"], gpus=case["gpus"])
    step = case.get("step", 0.1)
    plan["off"] = ratios(step or 0.25)
    plan["model"] = dict(plan["model"], num_hidden_layers=case["layers"])
    raw = build(seed, plan)
    raw["tuning"].update(tuning_granularity=case.get("granularity", "inter-stage"), sample_size=case.get("samples", 1),
                         activation_checkpointing_tuning_enabled=case.get("ckpt_tuning", True))
    if not step:
        del raw["tuning"]["search_space"]
    return raw


def _strategy(case, rng):
    """A strategy of equal meshes with the offload ratios and checkpoint counts of the seed."""
    S, L = case["stages"], case["layers"]
    layers = [L // S + (1 if i < L % S else 0) for i in range(S)]
    n = case["nodes"] // S
    row = lambda: [4, n * 8, 1, 0, 0, 1] + [round(float(x), 2) for x in rng.uniform(0.1, 0.9, size=4)]
    return dict(enabled=True, layer_partitions=layers, device_assignment=[[n, 8]] * S,
                gradient_checkpointing=[int(rng.integers(0, l + 1)) for l in layers],
                gradient_accumulation_steps=case["grad_accum"], stage_strategies=[row() for _ in range(S)],
                pre_post_strategy="preset", pre_post_strategy_array=[4, n * 8, 1, 0, 0, 1, 0, 0, 0, 0])


def prepare(case, seed):
    if case["kind"] == "analyze":
        # micro-batches of four on every GPU of a stage
        raw = _raw(dict(case, batch=4 * case["nodes"] * case["gpus"] // case["stages"] * case["grad_accum"]), seed)
        raw["strategy"] = _strategy(case, np.random.default_rng(seed))
        return case, MistConfig(raw), None
    config = MistConfig(_raw(case, seed))
    return case, config, LayerTables(config) if case["kind"] != "tune" else None


def run(state):
    case, config, layers = state
    if case["kind"] == "tune":
        cost, solution = tune(config)
        grad_accum, stages = (0, []) if solution is None else solution
        # (layer range, mesh, checkpoints, policy) and strategy row of each stage; -1 behind the last one
        where = np.full((case["layers"], 6), -1, dtype=np.int64)
        rows = np.full((case["layers"], 10), -1.0)
        for i, ((span, mesh, ckpt, policy), row) in enumerate(stages):
            where[i], rows[i] = (*span, *mesh, ckpt, policy), row
        return dict(cost=float(cost), grad_accum=int(grad_accum), stages=where, strategies=rows)
    if case["kind"] == "analyze":
        total, stable, delta, peaks = analyze(config)
        return dict(total=float(total), stable=np.array(stable, dtype=np.float64),
                    delta=np.array(delta, dtype=np.float64), peaks=np.array(peaks, dtype=np.float64))
    L = case["layers"]
    meshes = _get_device_mesh_candidates(case["nodes"], case["gpus"], contiguous_inter_node=False)
    if case["kind"] == "tables":
        grad_accums = _get_grad_accumu_steps_candidates(case["batch"])
        tables = intra_stage_tune(layers, L, meshes, grad_accums, case["tp"], config, sample_size=case["samples"]).device
        return dict(stable=tables.stable, delta=tables.delta, index=tables.index)
    micro_batches = min(case["grad_accum"], L, case["nodes"] * case["gpus"])
    return batched_tune_best_latency_for_stage(
        layers, layers, layers, range(micro_batches), range(1, L + 1), range(L + 1), case["nodes"], case["gpus"],
        case["grad_accum"], config, tp_size=case["tp"], sample_size=case["samples"])


def work(case):
    """Every strategy row's latency and memory terms once (36 interference evaluations and the
    sums over them, about 500 operations), and one evaluation (about 60) and 20 bytes for each cell
    of a table that comes back."""
    if case["kind"] == "analyze":
        return dict(bytes=400.0 * case["stages"], flops=600.0 * case["stages"])
    config = MistConfig(_raw(case, 0))
    factory = SearchSpaceFactory(config, LayerTables(config).constraint)
    L = case["layers"]
    meshes = _get_device_mesh_candidates(case["nodes"], case["gpus"], contiguous_inter_node=False)
    grad_accums = _get_grad_accumu_steps_candidates(case["batch"])
    tps = tp_candidates(config) if case["kind"] == "tune" else [case["tp"]]
    if case["kind"] == "stage":
        meshes, grad_accums = [(case["nodes"], case["gpus"])], [case["grad_accum"]]
    rows = sum(factory.make(n, m, case["batch"], G, tp).n_rows for tp in tps for G in grad_accums for n, m in meshes)
    if case["kind"] == "tune":
        return dict(bytes=1e4, flops=500.0 * rows)
    P = min(max(n * m for n, m in meshes), L, max(grad_accums))
    cells = len(meshes) * len(grad_accums) * (2 * P * L * (L + 1) + L * (L + 1) + L + 1) * case["samples"]
    return dict(bytes=(20.0 if case["kind"] == "tables" else 96.0) * cells, flops=500.0 * rows + 60.0 * cells)


def tolerance(case):
    """Sums, quotients and comparisons in float64 with a fixed order, first index on ties."""
    return "exact"
