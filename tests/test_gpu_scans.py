"""The exclusive scans at the sizes where they change form: one block, two
launches, three launches, and the edges of their tiles.  Seen through the cell
starts (64-bit packed counts) of lists of that many cells, and through the ghost
starts of that many particles."""
import numpy as np
import pytest
import torch

from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


# cells along x; rows of (cells + 2) x 3 x 3 with the padding
@pytest.mark.parametrize("cells", [1, 453, 454, 1818, 1819, 1820, 1821, 1900, 233015, 233016, 233100])
def test_cell_starts(cells):
    rng = np.random.default_rng(cells)
    n = 5000
    pos = torch.from_numpy(rng.random((3, n)) * np.array([[float(cells)], [1.0], [1.0]])).float().cuda()
    out = torch.empty_like(pos)
    cl = vdm.CellListGPU(torch.float32, (0.0,) * 3, (float(cells), 1.0, 1.0), (cells, 1, 1),
                         vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION, 1.0)
    cl.construct(pos, n, n - 7, out)
    a = cl.arrays()
    cx = torch.clamp(torch.floor(pos[0]).long() + 1, max=cells + 1)
    cell = cx + (cells + 2) * (1 + 3 * 1)
    total = (cells + 2) * 9
    want = torch.zeros(total + 1, dtype=torch.long, device="cuda")
    want[1:] = torch.cumsum(torch.bincount(cell, minlength=total), 0)
    assert torch.equal(a["cell_start"].long(), want)
    want[1:] = torch.cumsum(torch.bincount(cell[: n - 7], minlength=total), 0)
    assert torch.equal(a["dom_start"].long(), want)
    assert torch.equal(a["s2n"].long(), torch.argsort(cell, stable=True))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 4096, 4097, 16383, 16384, 16385, 20480, 20481, 2097151, 2097152,
                               2097153, 2200000])
def test_ghost_starts(n):
    pos = torch.rand((3, n), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (1, 1, 1), 0.05, dtype=torch.float32, capacity=2 * n + 64)
    vd.pos[:, :n] = pos
    G = vd.ghost_get()
    lo, hi = (pos < 0.05).long(), (pos >= 1.0 - 0.05).long()
    per = (1 + lo + hi).prod(dim=0) - 1  # images of each particle
    assert abs(G - int(per.sum())) <= 0
    pid, _ = vd.ghost_opart()
    assert torch.equal(pid.long(), torch.repeat_interleave(torch.arange(n, device="cuda"), per))
