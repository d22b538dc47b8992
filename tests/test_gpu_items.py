"""Target items where their grouping can go wrong: rows of more cells than one
round of the item kernel covers (1024), gaps of more cells than an item may
span (8) and than a block holds (16), cells of 63, 64, 65 and more particles,
items that end inside a cell.  Neighbour counts over the cell tiles and Verlet
rows of every domain particle against a direct search."""
import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu

# (first cell, particles per cell over consecutive cells)
PATTERNS = {
    "gaps": [(0, [1]), (8, [2]), (17, [3, 0, 0, 4]), (40, [5, 0, 0, 0, 0, 0, 0, 6]), (56, [7, 0, 0, 0, 0, 0, 0, 0, 8]),
             (1020, [9, 1, 1, 1, 1, 1, 1, 1, 1, 2])],
    "full": [(3, [63, 1, 64, 65, 0, 128, 129, 2]), (15, [40] * 20), (1000, [30, 33, 31] * 10)],
    "dilute": [(k, [1]) for k in range(2, 1095, 3)],
}


def dense(rng):
    """Cells of thousands: rows of more mask words than an item tabulates, words
    full of hits and words without any."""
    p = np.concatenate([rng.random((3, 2700)) * 0.4 + np.array([[10.0 + k], [1.0], [1.0]]) for k in range(3)], axis=1)
    return np.concatenate([p, rng.random((3, 100)) * np.array([[30.0], [3.0], [3.0]])], axis=1)


@pytest.mark.parametrize("box_nn", [1, 2, 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("r", [0.999, 0.3])
def test_rows_of_dense_cells(r, dtype, box_nn):
    npd = np.float32 if dtype == torch.float32 else np.float64
    pos = np.ascontiguousarray(dense(np.random.default_rng(2)).astype(npd))
    n = pos.shape[1]
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (30.0, 3.0, 3.0), (0, 0, 0), 0.5, dtype=dtype)
    vd.pos[:, :n] = torch.from_numpy(pos).cuda()
    opt = vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION
    cl = vd.updateCellListGPU(vd.getCellListGPU(1.0 / box_nn, opt, NNIteratorBox=box_nn))
    vl = vdm.VerletListGPU()
    vl.build(cl, vd.pos, r)
    off, nbr = (t.cpu().numpy() for t in vl.arrays())
    s2n = cl.arrays()["s2n"].cpu().numpy()
    dom = cl.arrays()["dom"].cpu().numpy()
    rng = np.random.default_rng(3)
    for k in np.concatenate([np.arange(40), rng.integers(0, n, 400), [n - 1]]):
        i = s2n[dom[k]]
        d = pos - pos[:, i:i + 1]
        near = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2] < npd(r) * npd(r)
        row = nbr[off[k]:off[k + 1]]
        assert np.all(np.diff(row) > 0)
        np.testing.assert_array_equal(np.sort(s2n[row]), np.flatnonzero(near))


@pytest.mark.parametrize("rel", [0.0, 2.0 ** -23, 2.0 ** -20, 2.0 ** -17])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_distances_at_the_radius(dtype, rel):
    """Pairs whose distance is the radius to within rel (up to and past what the
    FP32 products can decide): every decision is the exact test's."""
    npd = np.float32 if dtype == torch.float32 else np.float64
    rng = np.random.default_rng(6)
    r = 0.5
    c = rng.random((3, 300)) * 2.0 + 1.0
    v = rng.standard_normal((3, 300))
    v *= r * (1.0 + rel * rng.uniform(-1.0, 1.0, 300)) / np.linalg.norm(v, axis=0)
    pos = np.ascontiguousarray(np.concatenate([c, c + v], axis=1).astype(npd))
    n = pos.shape[1]
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (4.0,) * 3, (0, 0, 0), r, dtype=dtype)
    vd.pos[:, :n] = torch.from_numpy(pos).cuda()
    cl, vl = vd.getVerletGPU(r, sub=1)
    off, nbr = (t.cpu().numpy() for t in vl.arrays())
    s2n = cl.arrays()["s2n"].cpu().numpy()
    dom = cl.arrays()["dom"].cpu().numpy()
    for k in range(n):
        d = pos - pos[:, s2n[dom[k]]][:, None]
        near = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2] < npd(r) * npd(r)
        np.testing.assert_array_equal(np.sort(s2n[nbr[off[k]:off[k + 1]]]), np.flatnonzero(near))


@pytest.mark.parametrize("box_nn", [1, 2])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("pattern", sorted(PATTERNS))
def test_counts_and_rows(pattern, dtype, box_nn):
    rng = np.random.default_rng(9)
    pos = []
    for c0, per in PATTERNS[pattern]:
        for k, m in enumerate(per):
            p = rng.random((3, m))
            p[0] += c0 + k
            p[1:] = p[1:] * 2.0 + 0.5  # a few x-rows
            pos.append(p)
    npd = np.float32 if dtype == torch.float32 else np.float64
    pos = np.ascontiguousarray(np.concatenate(pos, axis=1)[:, rng.permutation(sum(p.shape[1] for p in pos))].astype(npd))
    n = pos.shape[1]
    r = 0.999
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1100.0, 3.0, 3.0), (0, 0, 0), 0.5, dtype=dtype)
    vd.pos[:, :n] = torch.from_numpy(pos).cuda()
    # the quantised stream holds rows of up to 2048 cells
    quant = vdm.CL_QUANT if box_nn == 1 else 0
    opt = vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION | quant
    cl = vd.updateCellListGPU(vd.getCellListGPU(1.0 / box_nn, opt, NNIteratorBox=box_nn))
    n2s = cl.arrays()["n2s"].long()[:n]
    d = pos[:, :, None] - pos[:, None, :]  # FP32 differences as the Verlet test rounds them
    d2 = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]
    near = d2 < npd(r) * npd(r)
    x = pos.astype(np.float64)
    e = x[:, :, None] - x[:, None, :]
    want = ((e[0] ** 2 + e[1] ** 2) + e[2] ** 2 < r * r).sum(axis=1) - 1
    for prec in (L.OFP_PREC_F64, L.OFP_PREC_F32C) if quant else (L.OFP_PREC_F64,):
        nn = torch.zeros(vd.cap, dtype=torch.int32, device="cuda")
        prm = L.LJParams(r, 0.01, 1.0)
        L.call("ofp_pair_lj", cl.h, None, vd.pos.data_ptr(), vd.cap, prec, prm, None, None, None, None, nn.data_ptr(),
               vdm._stream())
        np.testing.assert_array_equal(nn[n2s].cpu().numpy(), want)
    vl = vdm.VerletListGPU()
    vl.build(cl, vd.pos, r)
    off, nbr = (t.cpu().numpy() for t in vl.arrays())
    s2n = cl.arrays()["s2n"].cpu().numpy()
    dom = cl.arrays()["dom"].cpu().numpy()
    for k in range(n):
        row = nbr[off[k]:off[k + 1]]
        assert np.all(np.diff(row) > 0)
        np.testing.assert_array_equal(np.sort(s2n[row]), np.flatnonzero(near[s2n[dom[k]]]))
