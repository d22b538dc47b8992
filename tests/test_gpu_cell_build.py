"""The cell-list build at the sizes where it changes form: the edges of its tiles
(1024 keys, 4096 from 2^20 particles), the table summed in the scatter (up to 32
tiles), with the sums of chunks of them (up to 2048) or in kernels of its own,
and input in cell order (the order check's own build) against input nearly in
that order and in none.  Exact: permutations, cell
starts, domain order, sorted positions and planes."""
import pytest
import torch

from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu

TILES = [1, 1023, 1024, 1025, 2049, 32 * 1024, 32 * 1024 + 1, 300001, (1 << 20) - 1, 1 << 20, (1 << 20) + 4097,
         2048 * 4096, 2048 * 4096 + 1]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", TILES)
def test_cell_build(n, dtype):
    # (cells per side, order of the input); 2 cells: one pass; 31: two; 41: 3 passes
    for side, order in ((2, "none"), (31, "none"), (31, "exact"), (31, "near"), (41, "none"), (41, "exact")):
        gen = torch.Generator(device="cuda").manual_seed(n + side)
        pos = torch.rand((3, n), generator=gen, device="cuda", dtype=dtype) * side
        total = (side + 2) ** 3

        def cells(p):
            c = torch.clamp(torch.floor(p).long() + 1, max=side + 1)
            return c[0] + (side + 2) * (c[1] + (side + 2) * c[2])

        if order != "none":
            pos = pos[:, torch.argsort(cells(pos), stable=True)].contiguous()
            if order == "near" and n > 2:
                i = n - 2  # one exchanged pair, at the end of the input
                pos[:, [0, i]] = pos[:, [i, 0]]
        gm = n - n // 5
        out = torch.empty_like(pos)
        cl = vdm.CellListGPU(dtype, (0.0,) * 3, (float(side),) * 3, (side,) * 3,
                             vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION, 1.0)
        for _ in range(2):  # the second build starts from used buffers
            cl.construct(pos, n, gm, out)
            a = cl.arrays()
            c = cells(pos)
            perm = torch.argsort(c, stable=True)
            assert torch.equal(a["s2n"].long(), perm), (side, order)
            assert torch.equal(a["n2s"].long()[perm], torch.arange(n, device="cuda")), (side, order)
            want = torch.zeros(total + 1, dtype=torch.long, device="cuda")
            want[1:] = torch.cumsum(torch.bincount(c, minlength=total), 0)
            assert torch.equal(a["cell_start"].long(), want), (side, order)
            want[1:] = torch.cumsum(torch.bincount(c[:gm], minlength=total), 0)
            assert torch.equal(a["dom_start"].long(), want), (side, order)
            assert torch.equal(out, pos[:, perm]), (side, order)
