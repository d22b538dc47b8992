"""SPH passes over Verlet rows at the row lengths where their steps end (a row's
whole steps run without masks, its last partial step with them): isolated
clumps of m particles, every row m entries long, against the cubic spline
summed in FP64 on the host.  Coincident particles are neighbours with W(0) and
no force; a particle whose position is not a number keeps W(0) alone."""
import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 15, 16, 17, 48, 63, 64, 65, 127, 128, 129, 200)
H = 0.05


def w_dw(q):
    w = np.where(q < 1, 1 - 1.5 * q ** 2 + 0.75 * q ** 3, np.where(q < 2, 0.25 * (2 - q) ** 3, 0.0))
    dw = np.where(q < 1, -3 * q + 2.25 * q ** 2, np.where(q < 2, -0.75 * (2 - q) ** 2, 0.0))
    return w, dw


def clumps(dtype, lo, hi, coincident):
    """A clump of every size, each inside a ball of diameter 1.05 x 2h (some pairs
    beyond the cut-off, all inside the Verlet radius 1.1 x 2h)."""
    rng = np.random.default_rng(3)
    out, first = [], [0]
    for k, m in enumerate(SIZES):
        c = np.array([k % 3, (k // 3) % 3, k // 9]) * 0.3 + 0.2
        v = rng.standard_normal((3, m))
        v *= (rng.random(m) ** (1 / 3) * 0.5 * 2.1 * H) / np.linalg.norm(v, axis=0)
        p = c[:, None] + v
        if coincident and m > 4:
            p[:, 1] = p[:, 0]
            p[:, m - 1] = p[:, m // 2]
        out.append(p)
        first.append(first[-1] + m)
    return np.ascontiguousarray(np.concatenate(out, axis=1).astype(dtype)), first


@pytest.mark.parametrize("coincident", [False, True])
@pytest.mark.parametrize("box", [(1.0, 1.0, 1.2), (1.0, 1.03, 1.21)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("prec", [L.OFP_PREC_F64, L.OFP_PREC_F32C])
def test_rows_of_every_length(prec, dtype, box, coincident):
    pos, first = clumps(dtype, (0.0,) * 3, box, coincident)
    n = pos.shape[1] + 1
    pos = np.concatenate([pos, np.full((3, 1), np.nan, dtype)], axis=1)
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    odt = torch.float64 if prec == L.OFP_PREC_F64 else torch.float32
    r = 2.2 * H
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, box, (0, 0, 0), r, dtype=tdt)
    vd.pos[:, :n] = torch.from_numpy(pos).cuda()
    cl, vl = vd.getVerletGPU(r, vdm.CL_NON_SYMMETRIC | vdm.CL_QUANT)
    off, _ = vl.arrays()
    n2s = cl.arrays()["n2s"].long()[:n]
    rho = torch.zeros(vd.cap, dtype=torch.float64, device="cuda")
    prm = L.SPHParams(H, 0.7, 1000.0, 10.0)
    st = vdm._stream()
    L.call("ofp_sph_density", cl.h, vl.h, vd.pos.data_ptr(), vd.cap, prec, prm, rho.data_ptr(), st)
    rng = np.random.default_rng(4)
    pt = rng.random(n)
    ptd = torch.zeros(vd.cap, dtype=odt, device="cuda")
    ptd[n2s] = torch.from_numpy(pt).to(odt).cuda()
    F = torch.zeros((3, vd.cap), dtype=odt, device="cuda")
    L.call("ofp_sph_force", cl.h, vl.h, vd.pos.data_ptr(), vd.cap, prec, prm, ptd.data_ptr(), F[0].data_ptr(),
           F[1].data_ptr(), F[2].data_ptr(), st)
    rho, F = rho[n2s].cpu().numpy(), F[:, n2s].double().cpu().numpy()
    lens = np.sort((off[1:] - off[:-1]).cpu().numpy())
    assert list(lens) == sorted([0] + [m for m in SIZES for _ in range(m)])
    a = 0.7 / (np.pi * H ** 3)
    pt = ptd[n2s].double().cpu().numpy()
    x = pos.astype(np.float64)
    ref_r, ref_f = np.zeros(n), np.zeros((3, n))
    for b, e in zip(first[:-1], first[1:]):
        d = x[:, b:e, None] - x[:, None, b:e]
        dist = np.sqrt((d ** 2).sum(axis=0))
        w, dw = w_dw(dist / H)
        ref_r[b:e] = a * w.sum(axis=1)
        c = -a / H * (pt[b:e, None] + pt[None, b:e]) * np.where(dist > 0, dw / np.where(dist > 0, dist, 1.0), 0.0)
        ref_f[:, b:e] = (c[None] * d).sum(axis=2)
    ref_r[n - 1] = a
    # FP64: rounding of sums of up to 200 terms; FP32C: the records' quantum
    # (r / 2^28 per coordinate) and the FP32 stores
    tr, tf = (1e-13, 1e-13) if prec == L.OFP_PREC_F64 else (1e-7, 1e-6)
    assert np.all(np.abs(rho - ref_r) <= tr * ref_r)
    assert np.all(F[:, n - 1] == 0.0) and np.isfinite(F).all()
    mag = np.sqrt((ref_f ** 2).sum(axis=0))
    err = np.sqrt(((F - ref_f) ** 2).sum(axis=0))
    assert np.all(err <= tf * np.maximum(mag, np.sqrt((mag ** 2).mean())))
