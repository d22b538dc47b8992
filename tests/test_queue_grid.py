"""Launches that draw from the work queues bring a wave to every queue, however few
blocks were asked for; larger grids stay as they are."""
import ctypes as C

import pytest

from openfpm_pdata_amd import _lib as L


@pytest.mark.parametrize("waves", [1, 2, 3, 4, 8, 16])
def test_every_queue_has_a_wave(waves):
    grid, queues = C.c_uint(), C.c_uint()
    for blocks in (1, 2, 7, 15, 16, 17, 63, 64, 2048):
        L.call("ofp_test_queue_grid_", blocks, waves, C.byref(grid), C.byref(queues))
        drawn = {(b * waves + w) % queues.value for b in range(grid.value) for w in range(waves)}
        assert drawn == set(range(queues.value))
        assert grid.value >= blocks and (grid.value == blocks or blocks * waves < queues.value)
