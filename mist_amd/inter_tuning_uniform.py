"""Uniform inter-stage search: drop-in for the reference's
``mist/analyzer/inter_tuning_uniform.py`` (``inter_stage_tune`` :120-258,
``inter_stage_tune_with_fixed_inter_partition`` :261-397).

Layers and devices are split evenly over the stages, so the search is a few hundred table
look-ups per stage count; one launch does them where the tables are (``mist_uniform_search``;
sample slot 0 only, like the reference) and a few KB of totals come back.  Tables in host memory
are searched by the loops below.  Stage latency is ``stable + delta / G`` evaluated in float64: the
reference adds numpy float32 scalars to a python-int quotient, which numpy 1.24 promotes to float64.
"""
from __future__ import annotations

import ctypes
from typing import List, Optional

import numpy as np
import torch

from . import _lib
from .config import MistConfig
from .inter_tuning import get_solution_from_intra_stage_tuner_output
from .intra_tuning import IntraStageTunerOutput, to_device


def _uniform_layer_partition(num_layers: int, num_stages: int) -> List[int]:
    """inter_tuning_uniform.py:95-102: remainder layers go to the last stages."""
    per_stage = num_layers // num_stages
    partition = [per_stage] * num_stages
    for i in range(num_layers % num_stages):
        partition[-i - 1] += 1
    return partition


def _uniform_device_mesh_partition(num_stages: int, num_nodes: int, num_gpus_per_node: int):
    """inter_tuning_uniform.py:105-120."""
    if num_nodes > num_stages:
        if num_nodes % num_stages != 0:
            return None
        return num_nodes // num_stages, num_gpus_per_node
    if num_stages % num_nodes != 0 or num_gpus_per_node % (num_stages // num_nodes) != 0:
        return None
    return 1, num_gpus_per_node // (num_stages // num_nodes)


def cells_wanted(num_layers: int, num_nodes: int, num_gpus_per_node: int):
    """What the uniform search reads of the intra-stage tables of a (G, mesh) group, for
    ``IntraStageTuner.cells_wanted``: a mesh is read for the one stage count S whose even split of
    the cluster it is, there for L // S layers (and one more where the layers do not divide) and
    the pre-saved micro-batch values 0..S-1."""
    num_devices = num_nodes * num_gpus_per_node

    def wanted(G: int, mesh):
        n, m = mesh
        if n * m <= 0 or num_devices % (n * m) != 0:
            return None
        S = num_devices // (n * m)
        if S > num_layers or _uniform_device_mesh_partition(S, num_nodes, num_gpus_per_node) != mesh:
            return None
        return num_layers // S, -(-num_layers // S), S

    return wanted


def inter_stage_tune_with_fixed_inter_partition(
    num_layers: int,
    num_stages: int,
    layer_partition: List[int],
    device_mesh_index: int,
    gradient_accumulation_steps_candidates: List[int],
    gradient_accumulation_steps_index_candidates: List[int],
    tables,
    all_gradient_accumulation_steps: List[int],
    activation_checkpointing_tuning_enabled: bool,
    simple_activation_checkpointing_tuning_enabled: bool = False,
):
    """inter_tuning_uniform.py:261-397.  ``tables`` = (stable, delta) x 4 variants, float32;
    ``all_gradient_accumulation_steps[g]`` is the G of table index g."""
    (cs, cs_pre, cs_post, cs_nopp), (cd, cd_pre, cd_post, cd_nopp) = tables
    partition = np.array(layer_partition)
    starts = np.cumsum(partition) - partition
    ends = np.cumsum(partition) - 1
    q = device_mesh_index

    def t_intra(g, stage_index, l_start, l_end, c):
        l = l_end - l_start + 1
        p = num_stages - stage_index - 1
        if l_start == 0 and l_end == num_layers - 1:
            stable, delta = cs_nopp[g, q, c, 0], cd_nopp[g, q, c, 0]
        elif l_start == 0:
            stable, delta = cs_pre[g, q, p, l - 1, c, 0], cd_pre[g, q, p, l - 1, c, 0]
        elif l_end == num_layers - 1:
            stable, delta = cs_post[g, q, l - 1, c, 0], cd_post[g, q, l - 1, c, 0]
        else:
            stable, delta = cs[g, q, p, l - 1, c, 0], cd[g, q, p, l - 1, c, 0]
        return np.float64(stable) + np.float64(delta) / all_gradient_accumulation_steps[g]

    best_cost, best_g, best_g_index, best_ckpt = np.inf, None, None, None
    for G, g in zip(gradient_accumulation_steps_candidates, gradient_accumulation_steps_index_candidates):
        if simple_activation_checkpointing_tuning_enabled:
            for c in range(0, min(layer_partition) + 1):
                lat = [t_intra(g, s, starts[s], ends[s], c) for s in range(num_stages)]
                if np.inf in lat:
                    continue
                total = max(lat) * (G - 1) + sum(lat)
                if total < best_cost:
                    best_cost, best_g, best_g_index, best_ckpt = total, G, g, [c] * num_stages
        else:
            lat, ckpts = [], []
            for s in range(num_stages):
                if not activation_checkpointing_tuning_enabled:
                    c_best = ends[s] - starts[s] + 1
                    t_best = t_intra(g, s, starts[s], ends[s], c_best)
                else:
                    c_best, t_best = None, np.inf
                    for c in range(ends[s] - starts[s] + 2):
                        t = t_intra(g, s, starts[s], ends[s], c)
                        if t < t_best:
                            t_best, c_best = t, c
                lat.append(t_best)
                ckpts.append(c_best)
            if np.inf in lat:
                continue
            total = max(lat) * (G - 1) + sum(lat)
            if total < best_cost:
                best_cost, best_g, best_g_index, best_ckpt = total, G, g, ckpts
    return best_cost, best_g, best_g_index, best_ckpt


def _search_on_device(num_layers, stage_counts, q_of, max_stages, results_list, mode):
    """``mist_uniform_search`` over the tables of ``results_list`` (slices of one batch or tables of
    their own): per result ``(totals[g, k], ckpts[g, k, stage], rows[g, k, stage])``."""
    lib = _lib.load()
    problems = np.array([(S, q) for S, q in zip(stage_counts, q_of)], dtype=np.int32)
    n_k, out = len(problems), []
    first = results_list[0]
    n_g = len(first.gradient_accumulation_steps_candidates)
    whole = (all(r.batch is first.batch and r.batch_index == i for i, r in enumerate(results_list))
             and first.batch.stable[0].shape[0] == len(results_list) * n_g)
    for tabs, results in ([(first.batch, results_list)] if whole else [(r.device, [r]) for r in results_list]):
        rows, Q, P1, L, _, samples = tabs.stable[0].shape
        dev = tabs.stable[0].device
        with torch.cuda.device(dev):
            Gs = np.array([G for r in results for G in r.gradient_accumulation_steps_candidates], dtype=np.int32)
            (d_in,) = to_device([np.concatenate((Gs, problems.reshape(-1)))], dev)
            n_cells = rows * n_k * max_stages
            d_out = torch.empty(2 * rows * n_k + 2 * n_cells, dtype=torch.int32, device=dev)
            at = d_out.data_ptr()
            struct = tabs.as_struct()
            _lib.check(lib.mist_uniform_search(
                ctypes.byref(struct), L, P1, samples, 0, Q, d_in.data_ptr(), rows,
                ctypes.c_void_p(problems.ctypes.data), d_in.data_ptr() + 4 * rows, n_k, max_stages, mode,
                at, at + 8 * rows * n_k, at + 8 * rows * n_k + 4 * n_cells,
                ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)), "mist_uniform_search")
            host = d_out.cpu().numpy()
        total = host[:2 * rows * n_k].view(np.float64).reshape(len(results), -1, n_k)
        ckpt, row = host[2 * rows * n_k:].reshape(2, len(results), -1, n_k, max_stages)
        out += list(zip(total, ckpt, row))
    return out


def inter_stage_tune_batch_uniform(
    num_layers: int,
    num_nodes: int,
    num_gpus_per_node: int,
    gradient_accumulation_steps_candidates: List[int],
    results_list: List[IntraStageTunerOutput],
    config: MistConfig,
):
    """``inter_stage_tune`` for several intra-stage results (the tensor-parallel candidates of one
    ``tune`` call) with one launch and one read-back."""
    for r in results_list:
        if not isinstance(r, IntraStageTunerOutput):
            raise TypeError(
                f"intra_stage_results must be an instance of IntraStageTunerOutput, got {type(r)}"
            )
    if any(r.batch.stable[0].device.type != "cuda" for r in results_list):
        return [_inter_stage_tune_on_host(num_layers, num_nodes, num_gpus_per_node,
                                          gradient_accumulation_steps_candidates, r, config)
                for r in results_list]
    tuning = config.tuning
    mode = 0 if tuning.activation_checkpointing_tuning_enabled else 1
    if tuning.tuning_granularity == "uniform-pp-simple-heuristic-mem-opt":
        mode = 2
    first = results_list[0]
    q_index = {q: i for i, q in enumerate(first.device_mesh_candidates)}
    P1 = first.batch.stable[0].shape[2]
    stage_counts, q_of, meshes = [], [], []
    for num_stages in range(1, num_layers + 1):
        if num_nodes * num_gpus_per_node % num_stages != 0:
            continue
        n, m = _uniform_device_mesh_partition(num_stages, num_nodes, num_gpus_per_node)
        q = q_index[(n, m)]
        if num_stages > max(P1, 1):
            raise IndexError(f"{num_stages} stages need {num_stages - 1} pre-saved micro-batches; "
                             f"the tables hold {P1} values")
        stage_counts.append(num_stages)
        q_of.append(q)
        meshes.append((n, m))
    found = _search_on_device(num_layers, stage_counts, q_of, max(stage_counts), results_list, mode)
    out = []
    for r, (total, ckpt, row) in zip(results_list, found):
        g_index = {G: i for i, G in enumerate(r.gradient_accumulation_steps_candidates)}
        g_of = [g_index[G] for G in gradient_accumulation_steps_candidates]
        best = (float("inf"), None, None)
        totals = total.tolist()
        for k in range(len(stage_counts)):  # stage counts ascending, then G in the given order; strict "<"
            for i, g in enumerate(g_of):
                if totals[g][k] < best[0]:
                    best = (totals[g][k], i, k)
        cost, i, k = best
        if k is None:
            out.append((float("inf"), None))
            continue
        S, g = stage_counts[k], g_of[i]
        layers = _uniform_layer_partition(num_layers, S)
        strategy = r.spaces[(g, q_of[k])].decode(row[g, k, :S].astype(np.int64)).tolist()
        solution, start = [gradient_accumulation_steps_candidates[i], []], 0
        for s in range(S):
            strategy[s][:6] = [int(x) for x in strategy[s][:6]]
            inter = ((start, start + layers[s] - 1), meshes[k], int(ckpt[g, k, s]), 0)
            solution[1].append((inter, tuple(strategy[s])))
            start += layers[s]
        out.append((cost, solution))
    return out


def inter_stage_tune(
    num_layers: int,
    num_nodes: int,
    num_gpus_per_node: int,
    gradient_accumulation_steps_candidates: List[int],
    intra_stage_results: IntraStageTunerOutput,
    config: MistConfig,
):
    """inter_tuning_uniform.py:120-258."""
    return inter_stage_tune_batch_uniform(
        num_layers, num_nodes, num_gpus_per_node, gradient_accumulation_steps_candidates,
        [intra_stage_results], config)[0]


def _inter_stage_tune_on_host(
    num_layers: int,
    num_nodes: int,
    num_gpus_per_node: int,
    gradient_accumulation_steps_candidates: List[int],
    intra_stage_results: IntraStageTunerOutput,
    config: MistConfig,
):
    """The same over tables in host memory."""
    r = intra_stage_results
    ckpt_tuning = config.tuning.activation_checkpointing_tuning_enabled
    simple = config.tuning.tuning_granularity == "uniform-pp-simple-heuristic-mem-opt"
    tables = (
        (r.costs_stable, r.costs_stable_with_pre, r.costs_stable_with_post, r.costs_stable_no_pp),
        (r.costs_delta, r.costs_delta_with_pre, r.costs_delta_with_post, r.costs_delta_no_pp),
    )
    all_G = list(r.gradient_accumulation_steps_candidates)
    g_index = {G: i for i, G in enumerate(r.gradient_accumulation_steps_candidates)}
    q_index = {q: i for i, q in enumerate(r.device_mesh_candidates)}
    g_indices = [g_index[G] for G in gradient_accumulation_steps_candidates]

    best = (float("inf"), None, None, None, None)
    for num_stages in range(1, num_layers + 1):
        if num_nodes * num_gpus_per_node % num_stages != 0:
            continue
        partition = _uniform_layer_partition(num_layers, num_stages)
        n, m = _uniform_device_mesh_partition(num_stages, num_nodes, num_gpus_per_node)
        cost, G, g, ckpts = inter_stage_tune_with_fixed_inter_partition(
            num_layers, num_stages, partition, q_index[(n, m)],
            gradient_accumulation_steps_candidates, g_indices, tables, all_G, ckpt_tuning, simple,
        )
        if cost < best[0]:
            best = (cost, G, g, num_stages, ckpts)
    best_cost, best_g, best_g_index, best_num_stages, best_ckpts = best
    if best_g is None:
        return float("inf"), None

    partition = _uniform_layer_partition(num_layers, best_num_stages)
    n, m = _uniform_device_mesh_partition(best_num_stages, num_nodes, num_gpus_per_node)
    q = q_index[(n, m)]
    starts = np.cumsum(partition) - partition
    ends = np.cumsum(partition) - 1
    solutions = [best_g, []]
    for s in range(best_num_stages):
        row = get_solution_from_intra_stage_tuner_output(
            r, num_layers, best_g_index, best_num_stages - s - 1, int(starts[s]), int(ends[s]), q,
            int(best_ckpts[s]), slot=0,
        ).tolist()
        row[:6] = [int(x) for x in row[:6]]
        inter = ((int(starts[s]), int(ends[s])), (n, m), int(best_ckpts[s]), 0)
        solutions[1].append((inter, tuple(row)))
    return float(best_cost), solutions
