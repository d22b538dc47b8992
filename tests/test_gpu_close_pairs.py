"""SPH forces of isolated pairs at separations from 1e-6 h to 1.5 h, where a pair is all
that a force is summed from.  Reference: the cubic spline's slope in extended precision
from the stored positions.  A force is a product of about ten rounded factors, among
them 1 - r/2h >= 1/4, whose rounding counts fourfold and twice: 6e-15 relative."""
import math

import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu

QS = (1e-6, 1e-5, 1e-4, 1e-3, 1e-2, 0.1, 0.5, 0.999, 1.0, 1.001, 1.5)


@pytest.mark.parametrize("walk", ["rows", "cells"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_forces(dtype, walk):
    h, mass = 0.05, 0.3
    rng = np.random.default_rng(8)
    npd = np.float32 if dtype == torch.float32 else np.float64
    m = 8  # pairs per edge, 0.25 apart
    c = (np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij")).reshape(3, -1) + 0.5) * 0.25
    k = c.shape[1]
    v = rng.standard_normal((3, k))
    v *= np.resize(QS, k) * h / np.linalg.norm(v, axis=0)
    pos = np.ascontiguousarray(np.concatenate([c, c + v], axis=1).astype(npd))
    n = 2 * k
    pt = rng.random(n) + 0.5
    r = 2.0 * h * (1.1 if walk == "rows" else 1.0)
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (2.0,) * 3, (0, 0, 0), r, dtype=dtype)
    vd.pos[:, :n] = torch.from_numpy(pos).cuda()
    cl, vl = vd.getVerletGPU(r)
    n2s = cl.arrays()["n2s"].long()[:n]
    pts = torch.zeros(vd.cap, dtype=torch.float64, device="cuda")
    pts[n2s] = torch.from_numpy(pt).cuda()
    F = torch.zeros((3, vd.cap), dtype=torch.float64, device="cuda")
    L.call("ofp_sph_force", cl.h, vl.h if walk == "rows" else None, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F64,
           L.SPHParams(h, mass, 1000.0, 10.0), pts.data_ptr(), F[0].data_ptr(), F[1].data_ptr(), F[2].data_ptr(),
           vdm._stream())
    got = F[:, n2s].cpu().numpy().astype(np.longdouble)
    x = pos.astype(np.longdouble)
    pl = pt.astype(np.longdouble)
    d = x[:, :k] - x[:, k:]
    rr = np.sqrt((d * d).sum(axis=0))
    q = rr / np.longdouble(h)
    slope = np.where(q < 1, (-3 + np.longdouble(2.25) * q) / np.longdouble(h),
                     np.longdouble(-0.75) * (2 - q) ** 2 / np.where(rr > 0, rr, 1))
    f = -np.longdouble(mass) / (np.longdouble(math.pi) * np.longdouble(h) ** 4) * (pl[:k] + pl[k:]) * slope * d
    size = np.sqrt((f * f).sum(axis=0))
    use = rr > 0  # (FP32 positions hold no separation of 1e-6 h at some places)
    assert use.sum() > k / 2
    for side, sign in ((slice(0, k), 1), (slice(k, n), -1)):
        err = np.sqrt(((got[:, side] - sign * f) ** 2).sum(axis=0))[use] / size[use]
        assert err.max() < 6e-15, err.max()
