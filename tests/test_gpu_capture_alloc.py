"""A captured call that allocates (capture mode relaxed, where hipMalloc is allowed)
while the library keeps a block of the size from a destroyed list."""
import threading

import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu

N, R, H = 20000, 0.06, 0.027


def verlet():
    x = np.random.default_rng(5).random((3, N)).astype(np.float32)
    vd = vdm.VectorDistGPU(N, (0.0,) * 3, (1.0,) * 3, (0, 0, 0), R, dtype=torch.float32)
    vd.pos[:, :N] = torch.from_numpy(x).cuda()
    cl, vl = vd.getVerletGPU(R, vdm.CL_NON_SYMMETRIC | vdm.CL_QUANT)
    return vd, cl, vl


def force(made, pterm, F):
    vd, cl, vl = made
    fp = vdm.planes_of(F)
    L.call("ofp_sph_force", cl.h, vl.h, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F32C, L.SPHParams(H, 0.1, 1000.0, 10.0),
           pterm.data_ptr(), fp[0][0], fp[1][0], fp[2][0], vdm._stream())


def test_first_force_pass_in_a_captured_call():
    a, b = verlet(), verlet()
    cap = a[0].cap
    pterm = torch.rand(cap, device="cuda") + 0.5
    want = torch.zeros((3, cap), device="cuda")
    force(a, pterm, want)
    torch.cuda.synchronize()
    del a  # its blocks stay with the library
    got = torch.zeros_like(want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="relaxed"):
        force(b, pterm, got)
    for _ in range(3):
        got.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_another_thread_allocates_during_a_capture():
    """The other thread's list takes kept blocks; the capture (of this thread's own
    calls) stands."""
    want = [t.clone() for t in verlet()[2].arrays()]
    x = torch.zeros(1000, device="cuda")
    lists = []
    torch.cuda.synchronize()

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            lists.append(vdm.VerletListGPU())
            lists[0].build(made[1], made[0].pos, R)
            torch.cuda.current_stream().synchronize()

    made = verlet()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        x.add_(1.0)
        t = threading.Thread(target=work)
        t.start()
        t.join()
        x.add_(1.0)
    g.replay()
    torch.cuda.synchronize()
    assert x[0].item() == 2.0
    for a, b in zip(want, lists[0].arrays()):
        assert torch.equal(a, b)
