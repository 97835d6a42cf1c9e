"""The library's assignment solver leaves out thresholds by their bounds; the oracle tries all in turn."""
import numpy as np
import pytest

from oracle import inter_mip
from tests.test_oracle_mip import _random_assignment_problem, _solve_c


@pytest.mark.parametrize("quantum", [0.5, 0.125, 1e-4])  # from mostly ties to none
@pytest.mark.parametrize("G", [1, 2, 3, 32])
def test_thresholds_left_out_change_nothing(G, quantum):
    rng = np.random.default_rng(G)
    solved = 0
    for trial in range(25):
        S, avg, P = int(rng.integers(1, 7)), int(rng.integers(1, 9)), int(rng.integers(1, 12))
        layers = list(range(max(avg - 3, 1), avg + 4))
        L = S * avg + int(rng.integers(-1, 2))
        if L < S or layers[-1] > L:
            continue
        choices, t_s, t_d = _random_assignment_problem(rng, S, layers, P, quantum, float(rng.choice([0.0, 0.3, 0.8])))
        for best_cost in (inter_mip.MAX_VALUE, 15.0, 3.0):
            want_cost, want_picks = inter_mip.solve(L, layers, choices, t_s, t_d, G, best_cost)
            cost, picks = _solve_c(L, layers, choices, t_s, t_d, G, best_cost)
            assert picks == want_picks and (picks is None or cost == want_cost), (trial, best_cost)
            solved += picks is not None
    assert solved > 10
