"""``cost_table_kernel`` at the row lengths where its shifts, its workgroups and its passes end."""
import pytest

import tests.test_gpu_inter as inter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L, P1", [(15, 2), (16, 2), (31, 2), (63, 2), (64, 2), (127, 2), (128, 2), (255, 2),
                                   (256, 2), (257, 2)])
def test_cost_tables_at_the_edges_of_a_row(L, P1):
    inter.test_cost_tables_and_running_minima_equal_numpy(L, P1, 1 / 8, 0.4)
