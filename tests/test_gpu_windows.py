"""Windows of threshold candidates walked on the device, at the sizes and value distributions where their sort
changes its way, against numpy and the host's walk."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CAPACITY, DISTINCT, CHUNK, LEAD = 32768, 16384, 48, 16


def _values(rng, name, n):
    """`n` stage costs in any order."""
    if name == "even":
        v = np.linspace(1.0, 2.0, n)
    elif name == "repeated":
        v = rng.choice(1.0 + rng.random(max(1, n // 20)), n)
    elif name == "half":  # as many different ones as are walked and one more, most of them twice
        v = np.tile(np.linspace(1.0, 2.0, DISTINCT + 1), 2)[:n]
    elif name == "random":
        v = 1.0 + rng.random(n)
    elif name == "equal":
        v = np.full(n, 1.5)
    elif name == "crowded":  # all but one in one bucket of equal width: the general sort
        v = np.concatenate([1.0 + rng.random(n - 1) * 1e-2, [1e6]])
    elif name == "wide":  # a span that float32 cannot hold
        v = np.concatenate([1.0 + rng.random(n - 2), [-3e38, 3e38]])
    elif name == "narrow":  # a few neighbouring floats: a width that float32 cannot invert
        v = 1e-38 + rng.integers(0, 3, n) * 1.5e-45
    else:
        v = np.exp(rng.normal(0.0, 1.0, n))
    return v.astype(np.float32)


@pytest.mark.parametrize("name, n", [
    ("even", 1), ("even", 2), ("even", 63), ("even", 1023), ("even", 1024), ("even", 1025), ("even", 4097),
    ("even", 16383), ("even", 16384), ("even", 16385), ("equal", 1), ("equal", 5000), ("crowded", 100), ("crowded", 129),
    ("crowded", 16384), ("wide", 3000), ("narrow", 40), ("skewed", 9000), ("repeated", 5), ("repeated", 5000),
    ("repeated", 16385), ("repeated", 32768), ("repeated", 32769), ("random", 20000), ("random", 32768), ("half", 32768),
])
def test_windows_of_any_size_and_spread_equal_the_host_walk(name, n):
    import torch

    from mist_amd import _lib

    rng = np.random.default_rng(n)
    values = _values(rng, name, n)
    lib, dev = _lib.load(), torch.device("cuda:0")
    tables = torch.full((3, n), float("inf"), dtype=torch.float32, device=dev)
    tables[rng.integers(0, 3, n), np.arange(n)] = torch.from_numpy(values).to(dev)
    costs = _lib.DpCosts()
    for v, field in enumerate(("costs", "costs_pre", "costs_post")):
        setattr(costs, field, tables[v].data_ptr())
        costs.g_stride[v] = n
    order = np.unique(values)
    lo = np.float32(-np.inf) if name == "wide" else np.float32(order[0] - max(1e-4, 1e-4 * abs(float(order[0]))))
    start = order[len(order) // 3]
    f = lambda x: torch.tensor([x], dtype=torch.float32, device=dev)
    zeros = lambda k: torch.zeros(k, dtype=torch.int32, device=dev)
    row, d_lo, d_hi, d_start = zeros(1), f(lo), f(np.float32(3.4e38)), f(start)
    scratch, counts, kept = torch.empty(CAPACITY, device=dev), zeros(4), torch.empty(CAPACITY, device=dev)
    meta, inst_t, inst_row = zeros(8), torch.empty(CHUNK, device=dev), zeros(CHUNK)
    _lib.check(lib.mist_dp_windows_first_batch(
        ctypes.byref(costs), 1, row.data_ptr(), d_lo.data_ptr(), d_hi.data_ptr(), d_start.data_ptr(), 1e-6, CAPACITY, CHUNK,
        LEAD, scratch.data_ptr(), counts.data_ptr(), kept.data_ptr(), CAPACITY, meta.data_ptr(), inst_t.data_ptr(),
        inst_row.data_ptr(), None), "mist_dp_windows_first_batch")
    torch.cuda.synchronize()
    selected, above, status, n_kept, base, below, n_inst, first = meta.tolist()
    assert (selected, above) == (n, 0)
    if n > CAPACITY or len(order) > DISTINCT:
        assert status == 2
        return
    want = np.empty(len(order), dtype=np.float32)
    k = lib.mist_dp_window_begin(ctypes.c_void_p(order.ctypes.data), len(order), float(lo), 0, float(start), 1e-6,
                                 ctypes.c_void_p(want.ctypes.data))
    if k == _lib.DP_NO_START:
        assert status == 3
        return
    want = want[:k]
    if not (want >= start).any():
        assert status == 4
        return
    assert status == 0 and n_kept == k and below == int((want < start).sum())
    assert np.array_equal(kept.cpu().numpy()[base:base + k], want)
    at = [lib.mist_dp_first_batch_index(i, k - below, CHUNK, LEAD) for i in range(min(CHUNK, k - below))]
    assert n_inst == len(at) and np.array_equal(inst_t.cpu().numpy()[first:first + n_inst], want[below:][at])
    assert inst_row.tolist() == [0] * n_inst + [-1] * (CHUNK - n_inst)


def test_a_window_of_too_many_values_is_given_up_early(monkeypatch):
    """It costs less than the largest one that is walked."""
    import torch

    from mist_amd import _lib

    lib, least = _lib.load(), []
    call = lib.mist_dp_windows_first_batch

    def timed(*args):
        times = []
        for _ in range(10):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            status = call(*args)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        least.append(min(times))
        return status

    monkeypatch.setattr(lib, "mist_dp_windows_first_batch", timed)
    for n in (DISTINCT, CAPACITY):
        test_windows_of_any_size_and_spread_equal_the_host_walk("random", n)
    assert least[1] < least[0], least
