"""The FP32C density pass over Verlet rows without its 12-byte records (a captured
first call may not allocate them) against the pass with them, bit for bit, on every
replay; and beside a force pass of the same list on another stream."""
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 5000, 40001])
@pytest.mark.parametrize("box", [(1.0, 1.0, 1.0), (1.0, 1.1, 1.3)])
def test_density(n, box):
    h = 0.5 * (60.0 / n) ** (1.0 / 3.0) if n > 1000 else 0.05
    r = 2.2 * h
    gen = torch.Generator(device="cuda").manual_seed(n)
    pos = torch.rand((3, n), generator=gen, device="cuda") * torch.tensor(box, device="cuda")[:, None]
    prm = L.SPHParams(h, 0.7, 1000.0, 10.0)
    rho = []
    for captured in (False, True):
        vd = vdm.VectorDistGPU(n, (0.0,) * 3, box, (0, 0, 0), r, dtype=torch.float32)
        vd.pos[:, :n] = pos
        cl, vl = vd.getVerletGPU(r, vdm.CL_NON_SYMMETRIC | vdm.CL_QUANT)
        out = torch.zeros(vd.cap, dtype=torch.float64, device="cuda")

        def density(o):
            L.call("ofp_sph_density", cl.h, vl.h, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F32C, prm, o.data_ptr(),
                   vdm._stream())

        if captured:
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                density(out)
            for _ in range(3):
                out.zero_()
                torch.cuda.synchronize()
                g.replay()
                torch.cuda.synchronize()
                rho.append(out.clone())
        else:
            density(out)
            rho.append(out.clone())
            # beside force passes, which keep their own records in the list
            pt = torch.rand(vd.cap, generator=gen, device="cuda")
            F = torch.zeros((2, 3, vd.cap), device="cuda")

            def force(f):
                L.call("ofp_sph_force", cl.h, vl.h, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F32C, prm, pt.data_ptr(),
                       f[0].data_ptr(), f[1].data_ptr(), f[2].data_ptr(), vdm._stream())

            force(F[0])
            torch.cuda.synchronize()
            other = torch.cuda.Stream()
            for _ in range(5):
                both = torch.zeros_like(out)
                F[1].zero_()
                torch.cuda.synchronize()
                with torch.cuda.stream(other):
                    force(F[1])
                density(both)
                torch.cuda.synchronize()
                assert torch.equal(both, out) and torch.equal(F[0], F[1])
    for o in rho[1:]:
        assert torch.equal(o, rho[0])
