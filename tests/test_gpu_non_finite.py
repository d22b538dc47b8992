"""SPH passes with values and positions that are infinite or no number, over
Verlet rows and over cells: what lies beyond 2h, or at no distance that can be said,
adds nothing.  Reference: direct sums over the pairs within 2h, in FP64 (a sum of at
most n terms of about ten roundings each: relative to the sum of their sizes, 1e-13)."""
import math

import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu

MASS = 0.3


def setup(n, dtype, h, walk, scale=1.0, seed=1):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = (torch.rand((3, n), generator=gen, device="cuda", dtype=torch.float64) * scale).to(dtype)
    r = 2.0 * h * (1.3 if walk == "rows" else 1.0)
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (scale,) * 3, (0, 0, 0), r, dtype=dtype)
    vd.pos[:, :n] = x
    cl, vl = vd.getVerletGPU(r)
    return vd, cl, vl, gen


def squares(pos, n):
    x = pos[:, :n].double()
    d = x[:, :, None] - x[:, None, :]
    return d, d[0] * d[0] + d[1] * d[1] + d[2] * d[2]


def densities(vd, cl, vl, walk, h):
    rho = torch.zeros(vd.cap, dtype=torch.float64, device="cuda")
    L.call("ofp_sph_density", cl.h, vl.h if walk == "rows" else None, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F64,
           L.SPHParams(h, MASS, 1000.0, 10.0), rho.data_ptr(), vdm._stream())
    return rho


def check_densities(vd, cl, vl, walk, h, n):
    _, d2 = squares(vd.pos, n)
    q = torch.sqrt(d2) / h
    w = torch.where(q < 1, 1 - 1.5 * q ** 2 + 0.75 * q ** 3, 0.25 * (2 - q) ** 3)
    w = torch.where(d2 < 4 * h * h, w, torch.zeros_like(w))
    w.fill_diagonal_(1.0)
    want = w.sum(dim=1) * (MASS / (math.pi * h ** 3))
    got = densities(vd, cl, vl, walk, h)[:n]
    assert ((got - want).abs() <= 1e-13 * want).all()


@pytest.mark.parametrize("walk", ["rows", "cells"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
def test_values(value, dtype, walk):
    n, h = 900, 0.06
    vd, cl, vl, gen = setup(n, dtype, h, walk)
    pt = torch.rand(vd.cap, generator=gen, device="cuda", dtype=torch.float64) + 0.5
    pt[torch.arange(7, n, 150, device="cuda")] = value
    F = torch.full((3, vd.cap), 7.0, dtype=torch.float64, device="cuda")
    L.call("ofp_sph_force", cl.h, vl.h if walk == "rows" else None, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F64,
           L.SPHParams(h, MASS, 1000.0, 10.0), pt.data_ptr(), F[0].data_ptr(), F[1].data_ptr(), F[2].data_ptr(),
           vdm._stream())
    d, d2 = squares(vd.pos, n)
    r = torch.sqrt(d2)
    q = r / h
    s = torch.where(q < 1, (-3 + 2.25 * q) / h, -0.75 * (2 - q) ** 2 / r)
    c = (pt[:n, None] + pt[None, :n]) * s * (-MASS / (math.pi * h ** 4))
    near = (d2 < 4 * h * h) & (d2 > 0)
    t = torch.where(near[None], c[None] * d, torch.zeros_like(d))
    want, size = t.sum(dim=2), t.abs().sum(dim=2)
    got = F[:, :n]
    healthy = torch.isfinite(size)
    assert 0.5 * 3 * n < int(healthy.sum()) < 3 * n
    assert ((got - want).abs()[healthy] <= 1e-13 * size[healthy]).all()
    assert not torch.isfinite(got[~healthy]).any()


@pytest.mark.parametrize("walk", ["rows", "cells"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_a_value_without_neighbours(dtype, walk):
    """A particle on its own, and two in one place, have no force, whatever P/rho^2."""
    x = torch.tensor([[0.2, 0.7, 0.7], [0.5, 0.5, 0.5], [0.5, 0.5, 0.5]], device="cuda", dtype=dtype)
    h = 0.05
    vd = vdm.VectorDistGPU(3, (0.0,) * 3, (1.0,) * 3, (0, 0, 0), 2 * h, dtype=dtype)
    vd.pos[:, :3] = x
    cl, vl = vd.getVerletGPU(2 * h)
    pt = torch.full((vd.cap,), math.inf, device="cuda", dtype=torch.float64)
    F = torch.full((3, vd.cap), 7.0, dtype=torch.float64, device="cuda")
    L.call("ofp_sph_force", cl.h, vl.h if walk == "rows" else None, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F64,
           L.SPHParams(h, MASS, 1000.0, 10.0), pt.data_ptr(), F[0].data_ptr(), F[1].data_ptr(), F[2].data_ptr(),
           vdm._stream())
    assert torch.equal(F[:, :3], torch.zeros_like(F[:, :3]))


@pytest.mark.parametrize("walk", ["rows", "cells"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("value", [math.inf, math.nan])
def test_positions_since_the_build(value, dtype, walk):
    n, h = 900, 0.06
    vd, cl, vl, _ = setup(n, dtype, h, walk, seed=2)
    vd.pos[1, torch.arange(5, n, 90, device="cuda")] = value
    check_densities(vd, cl, vl, walk, h, n)


@pytest.mark.parametrize("walk", ["rows", "cells"])
@pytest.mark.parametrize("exponent", [0, -300, 300, 333])
def test_units_of_length(exponent, walk):
    scale = 2.0 ** exponent
    n, h = 500, 0.1 * scale
    vd, cl, vl, _ = setup(n, torch.float64, h, walk, scale, seed=3)
    check_densities(vd, cl, vl, walk, h, n)


@pytest.mark.parametrize("box", [(1.0, 1.0, 1.0), (1.0, 1.1, 1.3)])
@pytest.mark.parametrize("value", [math.inf, math.nan])
def test_values_fp32c_cells(value, box):
    """FP32C over cells: pairs at the cut-off to within what the candidate masks decide,
    a particle on its own and two in one place, all with the value.  (Over rows a
    particle's value reaches those whose rows hold it.)"""
    h, k = 0.05, 40
    gen = torch.Generator(device="cuda").manual_seed(6)
    g = torch.arange(4, device="cuda", dtype=torch.float64) * 0.25 + 0.125
    c = torch.stack(torch.meshgrid(g, g, g, indexing="ij")).reshape(3, -1)[:, :k]
    v = torch.randn((3, k), generator=gen, device="cuda", dtype=torch.float64)
    v = v / v.norm(dim=0) * 2.0 * h * (1.0 + torch.logspace(-7, -2, k, device="cuda", dtype=torch.float64))
    alone = torch.tensor([[0.9, 0.9, 0.9], [0.2, 0.8, 0.8], [0.2, 0.8, 0.8]], device="cuda", dtype=torch.float64)
    x = torch.cat([c, c + v, c[:, :1] + 0.02, alone], dim=1).float()
    n = x.shape[1]
    vd = vdm.VectorDistGPU(n, (-0.2,) * 3, tuple(b + 0.2 for b in box), (0, 0, 0), 2 * h, dtype=torch.float32)
    vd.pos[:, :n] = x
    cl = vd.updateCellListGPU(vd.getCellListGPU(2 * h, vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION | vdm.CL_QUANT))
    n2s = cl.arrays()["n2s"].long()[:n]
    bad = torch.zeros(n, dtype=torch.bool, device="cuda")
    bad[k:2 * k] = True
    bad[-3:] = True
    F = []
    for other in (value, 0.7):
        pt = torch.full((n,), 0.6, device="cuda")
        pt[bad] = other
        ps = torch.zeros(vd.cap, device="cuda")
        ps[n2s] = pt
        f = torch.full((3, vd.cap), 7.0, device="cuda")
        L.call("ofp_sph_force", cl.h, None, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F32C, L.SPHParams(h, MASS, 1000.0, 10.0),
               ps.data_ptr(), f[0].data_ptr(), f[1].data_ptr(), f[2].data_ptr(), vdm._stream())
        F.append(f[:, n2s])
    _, d2 = squares(x, n)
    near = (d2 < 4 * h * h * (1 + 1e-6)) & (d2 > 0)
    apart = ~(near & bad[None, :]).any(dim=1) & ~(bad & near.any(dim=1))
    assert int(apart[:k].sum()) > 10 and apart[-3:].all()
    assert torch.equal(F[0][:, apart], F[1][:, apart])
    assert torch.isfinite(F[0][:, apart]).all()
