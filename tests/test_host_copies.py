"""Strategy rows decoded a few at a time, and arrays packed into one copy, against the general ways."""
import numpy as np
import pytest


def test_a_few_rows_decode_like_many():
    from mist_amd.search_space import SearchSpace

    rng = np.random.default_rng(3)
    space = SearchSpace(par=rng.normal(size=(3, 6)), wo=(0.0, 0.5), go=(0.0, 0.25, 1.0), oo=(0.0, 1.0), ao=(0.0, 0.1, 0.2),
                        pair_wo=np.array([0, 0, 0, 1, 1], np.uint8), pair_go=np.array([0, 1, 2, 1, 2], np.uint8))
    every = np.arange(-1, space.n_rows)
    want = space.decode(every)
    for n in (1, 2, 16):
        for first in range(0, len(every) - n + 1, n):
            assert np.array_equal(space.decode(every[first:first + n]), want[first:first + n])
    assert np.array_equal(space.decode(np.array(4)), want[5]) and space.decode(np.zeros((2, 3), int)).shape == (2, 3, 10)
    assert space.decode(np.zeros((0,), int)).shape == (0, 10)
    with pytest.raises(AssertionError):
        space.decode(np.array([space.n_rows]))


def test_arrays_in_one_copy():
    import torch

    from mist_amd.intra_tuning import to_device

    arrays = [np.arange(5, dtype=np.int32), np.zeros(0, np.int64), np.arange(40, dtype=np.float64).reshape(5, 8)[:, ::2],
              np.zeros(3, dtype=[("a", "<i4"), ("b", "<f8")]), np.array([7], np.uint8)]
    for a, b in zip(arrays, to_device(arrays, torch.device("cpu"))):
        assert b.numpy().tobytes() == a.tobytes() and b.storage_offset() % 256 == 0
