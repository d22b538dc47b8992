"""The cell tiles' candidate masks at the sizes where their form changes: blocks of
32 and 64 targets, blocks of 32 and rounds of 256 and 384 candidates, stencils of 1
to 3 cells, cubic and other cells, FP32C and FP64; with particles that have moved
since the cells were built, and (FP64) one far outside the grid and one that is no
number.  Neighbour counts are exact, from the FP64 squares of the stored positions;
densities are those of the cubic spline summed in FP64 (relative 1e-12 in FP64; in
FP32C a separation is off by at most sqrt(3) 2^-28 of a cell, 1e-8 of the support,
and the spline's logarithmic derivative stays below 100 where it counts: 1e-6)."""
import math

import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 31, 32, 33, 64, 65, 255, 256, 257, 383, 384, 385, 700]


@pytest.mark.parametrize("spacing", [(1.0, 1.0, 1.0), (1.0, 1.125, 1.25)])
@pytest.mark.parametrize("nn", [1, 2, 3])
@pytest.mark.parametrize("prec,dtype", [(L.OFP_PREC_F64, torch.float64), (L.OFP_PREC_F64, torch.float32),
                                        (L.OFP_PREC_F32C, torch.float32)])
def test_counts_and_densities(prec, dtype, nn, spacing):
    r = 0.9 * nn - 0.5  # the stencil covers r and two moves of 0.2
    div = 9
    for m in SIZES:
        gen = torch.Generator(device="cuda").manual_seed(100 * m + nn)
        u = torch.rand((3, m), generator=gen, device="cuda", dtype=torch.float64)
        scale = torch.tensor([[3.0], [1.3], [1.3]], device="cuda", dtype=torch.float64)
        pos = (3.1 + u * scale).to(dtype)
        n = m
        if prec == L.OFP_PREC_F64:
            odd = torch.tensor([[500.0, math.nan], [4.0, 4.0], [4.0, 4.0]], device="cuda", dtype=dtype)
            pos = torch.cat([pos, odd], dim=1)
            n = m + 2
        pos = pos.contiguous()
        cl = vdm.CellListGPU(dtype, (0.0,) * 3, tuple(div * s for s in spacing), (div,) * 3,
                             vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION | vdm.CL_QUANT, r, box_nn=nn)
        out = torch.empty_like(pos)
        cl.construct(pos, n, n, out)
        if prec == L.OFP_PREC_F64:  # moved since the build
            move = torch.rand(out.shape, generator=gen, device="cuda", dtype=torch.float64) * 0.2
            out = (out.double() + move).to(dtype).contiguous()
        x = out.double()
        d = x[:, :, None] - x[:, None, :]
        d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        off = ~torch.eye(n, dtype=torch.bool, device="cuda")
        want = ((d2 < r * r) & off).sum(dim=1)
        odt = torch.float64 if prec == L.OFP_PREC_F64 else torch.float32
        F = torch.zeros((4, n), dtype=odt, device="cuda")
        cnt = torch.zeros(n, dtype=torch.int32, device="cuda")
        L.call("ofp_pair_lj", cl.h, None, out.data_ptr(), n, prec, L.LJParams(r, 0.2 * r, 1.0), F[0].data_ptr(),
               F[1].data_ptr(), F[2].data_ptr(), F[3].data_ptr(), cnt.data_ptr(), vdm._stream())
        assert torch.equal(cnt.long(), want), (m, nn)
        h = 0.5 * r
        rho = torch.zeros(n, dtype=torch.float64, device="cuda")
        L.call("ofp_sph_density", cl.h, None, out.data_ptr(), n, prec, L.SPHParams(h, 0.7, 1000.0, 10.0),
               rho.data_ptr(), vdm._stream())
        q = torch.sqrt(d2) / h
        w = torch.where(q < 1, 1 - 1.5 * q ** 2 + 0.75 * q ** 3, torch.where(q < 2, 0.25 * (2 - q) ** 3, 0.0))
        w = torch.where(off, torch.nan_to_num(w), torch.ones_like(w)).sum(dim=1) * (0.7 / (math.pi * h ** 3))
        rel = ((rho - w).abs() / w).max().item()
        assert rel < (1e-12 if prec == L.OFP_PREC_F64 else 1e-6), (m, nn, rel)
