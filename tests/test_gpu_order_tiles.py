"""The ordering by destination at the sizes where its tiles change: rounds of 64,
and the largest count for each tile size (the table of 16384 counts), by the map of
8 and of 3 ranks; exact against the oracle's order."""
import numpy as np
import pytest

from test_gpu_map import _check, _map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 1, 1)])
@pytest.mark.parametrize("n", [63, 64, 65, 116480, 116481, 131073, 262145, 349505, 1048577, 2100000])
def test_order(dims, n):
    m, pt, got, want = _map(dims, 1, (1, 0, 1), np.float32, n)
    _check(m, pt, got, want, n)
