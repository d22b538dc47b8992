"""Verlet rows of the item kernels, whose distances come from FP32 products on the
matrix cores, against a direct search in the list's own rounding: every decision is
the exact test's."""
import ctypes as C

import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


def check_rows(pos, r, cl, vl, npd):
    """Every row of vl against the squares of pos in npd's rounding."""
    rows = C.c_int(-1)
    L.call("ofp_vl_test_rows_", vl.h, C.byref(rows))
    assert rows.value == 0  # the item kernels built it
    off, nbr = (t.cpu().numpy() for t in vl.arrays())
    s2n = cl.arrays()["s2n"].cpu().numpy()
    dom = cl.arrays()["dom"].cpu().numpy()
    r2 = npd(r) * npd(r)
    for k in range(pos.shape[1]):
        d = pos - pos[:, s2n[dom[k]]][:, None]
        near = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2] < r2
        np.testing.assert_array_equal(np.sort(s2n[nbr[off[k]:off[k + 1]]]), np.flatnonzero(near), err_msg=str(k))


@pytest.mark.parametrize("sub", [1, 2])
@pytest.mark.parametrize("rel", [0.0, 2.0 ** -25, 2.0 ** -23, 2.0 ** -20, 2.0 ** -17])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_distances_at_the_radius(dtype, rel, sub):
    """Cells of 32 and more particles, every particle with a partner at the radius to
    within rel: undecided pairs in both blocks of candidates and both halves of an
    item's targets."""
    npd = np.float32 if dtype == torch.float32 else np.float64
    rng = np.random.default_rng(7)
    r, m = 0.5, 3000
    c = rng.random((3, m)) * 1.2 + 1.0
    v = rng.standard_normal((3, m))
    v *= r * (1.0 + rel * rng.uniform(-1.0, 1.0, m)) / np.linalg.norm(v, axis=0)
    pos = np.concatenate([c, c + v], axis=1)
    pos = np.ascontiguousarray(pos[:, rng.permutation(2 * m)].astype(npd))
    n = pos.shape[1]
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (3.5,) * 3, (0, 0, 0), r, dtype=dtype)
    vd.pos[:, :n] = torch.from_numpy(pos).cuda()
    cl, vl = vd.getVerletGPU(r, sub=sub)
    check_rows(pos, r, cl, vl, npd)


@pytest.mark.parametrize("n", [333, 999, 3000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_particles_beyond_their_cells(dtype, n):
    """Moved since the cells were built, further than the products' bound allows:
    every pair is tested in the list's own rounding.  The stencil spans the grid."""
    npd = np.float32 if dtype == torch.float32 else np.float64
    rng = np.random.default_rng(n)
    div, r = 4, 2.9
    pos = torch.from_numpy(np.ascontiguousarray((rng.random((3, n)) * div).astype(npd))).cuda()
    cl = vdm.CellListGPU(dtype, (0.0,) * 3, (float(div),) * 3, (div,) * 3,
                         vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION, 0.9, box_nn=3)
    out = torch.empty_like(pos)
    cl.construct(pos, n, n, out)
    s2n = cl.arrays()["s2n"].long()
    out = (out * 9.0).contiguous()
    pos = torch.empty_like(out)
    pos[:, s2n[:n]] = out
    vl = vdm.VerletListGPU()
    vl.build(cl, out, r)
    check_rows(pos.cpu().numpy(), r, cl, vl, npd)
