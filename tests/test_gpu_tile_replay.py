"""A captured pass over cell tiles, replayed after the cells were built anew from
another number of particles (the domain's stays, as when the ghosts change): it walks
the new cells' items."""
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gm", [3000, 40000, 300000])
def test_replay_after_a_rebuild(gm):
    cap = 4 * gm
    gen = torch.Generator(device="cuda").manual_seed(gm)
    pos = torch.rand((3, cap), generator=gen, device="cuda", dtype=torch.float64)
    div = round((gm / 8.0) ** (1.0 / 3.0))
    r = 1.0 / div
    cl = vdm.CellListGPU(torch.float64, (0.0,) * 3, (1.0,) * 3, (div,) * 3,
                         vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION, r)
    srt = torch.empty_like(pos)
    nn = torch.zeros((2, cap), dtype=torch.int32, device="cuda")

    def counts(out):
        L.call("ofp_pair_lj", cl.h, None, srt.data_ptr(), cap, L.OFP_PREC_F64, L.LJParams(r, 0.1 * r, 1.0), None, None,
               None, None, out.data_ptr(), vdm._stream())

    def build(n):
        cl.construct(pos, n, gm, srt)
        counts(nn[0])  # makes the items

    build(cap)  # buffers of the largest build, so that none is replaced later
    build(gm + 100)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        counts(nn[1])
    for n in (gm + 100, cap, gm, 2 * gm + 5, 3 * gm):
        nn.zero_()
        pos[:, :gm] = torch.roll(pos[:, :gm], 17, dims=1)
        build(n)
        g.replay()
        torch.cuda.synchronize()
        assert int(nn[0].sum()) > 0
        assert torch.equal(nn[0], nn[1]), n
