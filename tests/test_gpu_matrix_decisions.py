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


def scaled(dtype, scale, n=4000):
    """Particles in cells of 20 and more, and their lists' radius, in units of 1 / scale
    (a power of two: the same bits in the mantissas)."""
    rng = np.random.default_rng(11)
    p = np.concatenate([rng.random((3, n // 2)) * 3.4, 1.0 + rng.random((3, n // 2))], axis=1)
    npd = np.float32 if dtype == torch.float32 else np.float64
    pos = np.ascontiguousarray(p.astype(npd) * npd(scale))
    r = 0.6 * scale
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (3.5 * scale,) * 3, (0, 0, 0), r, dtype=dtype)
    vd.pos[:, :n] = torch.from_numpy(pos).cuda()
    return pos, r, vd, npd


EXPONENTS = (0, -40, -50, -63, -70, -100, -480, -505, 40, 60, 64, 100, 480, 505)


@pytest.mark.parametrize("dtype,exponent", [(torch.float64, e) for e in EXPONENTS] +
                         [(torch.float32, e) for e in EXPONENTS if abs(e) <= 100])
def test_units_of_length(dtype, exponent):
    """Lengths whose squares FP32 (and at the ends FP64) cannot hold: the rows are the
    direct search's in the positions' own arithmetic, the cell tiles' neighbour counts
    that of FP64."""
    pos, r, vd, npd = scaled(dtype, 2.0 ** exponent)
    n = pos.shape[1]
    cl, vl = vd.getVerletGPU(r, sub=1)
    with np.errstate(over="ignore", under="ignore"):
        check_rows(pos, r, cl, vl, npd)
    nn = torch.zeros(vd.cap, dtype=torch.int32, device="cuda")
    L.call("ofp_pair_lj", cl.h, None, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F64, L.LJParams(r, 0.1 * r, 1.0), None, None,
           None, None, nn.data_ptr(), vdm._stream())
    got = nn[cl.arrays()["n2s"].long()[:n]].cpu().numpy()
    x = pos.astype(np.float64)
    for i in range(n):
        d = x - x[:, i:i + 1]
        assert got[i] == np.count_nonzero((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2] < r * r) - 1, i
