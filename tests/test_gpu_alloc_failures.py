"""Allocations that a call can do without, refused as on a full device: the call goes
on without them and its results are those of an undisturbed call; one that it cannot
do without is an error of that call alone."""
from contextlib import contextmanager

import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import ensemble as E
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


@contextmanager
def refused(lo, hi, count):
    """The library's next `count` allocations of lo to hi bytes fail."""
    L.call("ofp_test_fail_alloc_", lo, hi, count)
    try:
        yield
    finally:
        L.call("ofp_test_fail_alloc_", 0, 0, 0)


def verlet(n=5000, r=0.09, seed=3):
    x = np.random.default_rng(seed).random((3, n)).astype(np.float32)
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (0, 0, 0), r, dtype=torch.float32)
    vd.pos[:, :n] = torch.from_numpy(x).cuda()
    cl, vl = vd.getVerletGPU(r, vdm.CL_NON_SYMMETRIC | vdm.CL_QUANT)
    return vd, cl, vl


def density(made, h=0.04):
    vd, cl, vl = made
    rho = torch.zeros(vd.cap, dtype=torch.float64, device="cuda")
    L.call("ofp_sph_density", cl.h, vl.h, vd.pos.data_ptr(), vd.cap, L.OFP_PREC_F32C, L.SPHParams(h, 0.1, 1000.0, 10.0),
           rho.data_ptr(), vdm._stream())
    return rho


def test_density_without_its_records():
    want = density(verlet())
    made = verlet()
    n = int(made[1].view().n_part)
    with refused(12 * n, 12 * (n + 2), 1):
        got = density(made)
    assert torch.equal(got, want)
    assert torch.equal(density(made), want)  # with them


@pytest.mark.parametrize("refusals", [1, 2])
def test_far_build_with_little_or_no_scratch(refusals):
    n = (1 << 22) + 12345
    gen = torch.Generator(device="cuda").manual_seed(4)
    pos = torch.rand((3, n), generator=gen, device="cuda")
    idx = torch.arange(n, device="cuda", dtype=torch.int32)
    out = []
    for k in (0, refusals):
        cl = vdm.CellListGPU(torch.float32, (0.0,) * 3, (1.0,) * 3, (78,) * 3, vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER,
                             1.0 / 78)
        srt, idx_s = torch.empty_like(pos), torch.empty_like(idx)
        with refused(30_000_000, 125_000_000, k):
            cl.construct(pos, n, n, srt, [(idx.data_ptr(), 4)], [(idx_s.data_ptr(), 4)])
        back = torch.empty_like(pos)
        cl.restore(vdm.planes_of(srt), vdm.planes_of(back))
        a = cl.arrays()
        out.append([a["s2n"].clone(), a["n2s"].clone(), srt, idx_s])
        assert torch.equal(back, pos)
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_a_refused_call_leaves_no_error_behind():
    made = verlet()
    with refused(1, 1 << 40, 1):
        with pytest.raises(L.OfpError):
            vdm.VerletListGPU().build(made[1], made[0].pos, 0.09)
    off, nbr = (t.clone() for t in made[2].arrays())
    made[2].build(made[1], made[0].pos, 0.09)
    for a, b in zip((off, nbr), made[2].arrays()):
        assert torch.equal(a, b)
    torch.cuda.synchronize()


def random_gas(n, seed=2):
    m = round(n ** (1.0 / 3.0)) + 1
    g = torch.Generator(device="cuda").manual_seed(seed)
    c = torch.randperm(m ** 3, generator=g, device="cuda")[:n]
    x = (torch.stack([c % m, (c // m) % m, c // (m * m)]).double() + 0.5) / m
    v = torch.randn((3, n), generator=g, device="cuda", dtype=torch.float64)
    ens = E.Ensemble([E.System(n, 1.6 / m, 0.8 / m, 1.0, 1.0)], torch.float32, E.Options(skin=0.1, sub=1, lanes=1))
    ens.set(x.float().contiguous(), v.float().contiguous())
    return ens


def test_far_run_without_its_cursors():
    n = (1 << 22) + 77
    out = []
    for k in (0, 1):
        ens = random_gas(n)
        ens.force_pass(L.OFP_PREC_F64)
        with refused(12288, 12288, k):
            ens.run(L.OFP_PREC_F64, 1e-7, 3)
        out.append(ens.get())
        del ens
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_forces_after_a_refused_run():
    """A run in another precision that fails before its steps leaves the forces of
    the last pass, each with its particle."""
    ens = random_gas(3000)
    want = ens.forces(L.OFP_PREC_F64)
    assert float(want.abs().max()) > 0
    with refused(1, 4096, 1):  # the other precision's tables
        with pytest.raises(L.OfpError):
            ens.run(L.OFP_PREC_F32C, 1e-7, 3)
    assert torch.equal(ens.get()[2], want)
    ens.run(L.OFP_PREC_F32C, 1e-7, 3)


@pytest.mark.parametrize("size", [1, 24])  # any first table, and the second one (24 bytes a system)
def test_tables_of_many_systems(size):
    S = 200
    gen = torch.Generator(device="cuda").manual_seed(9)
    x = torch.rand((3, 20 * S), generator=gen, device="cuda")
    systems = [E.System(20, 0.2, 0.02, 1.0, 1.0) for _ in range(S)]
    out = []
    for k in (0, 1):
        ens = E.Ensemble(systems, torch.float32, E.Options(skin=0.1, sub=1))
        ens.set(x)
        ens.rebuild()
        if k:
            lo, hi = (24 * S, 24 * S) if size == 24 else (24 * S + 1, 400 * S)
            with refused(lo, hi, 1):
                with pytest.raises(L.OfpError):
                    ens.force_pass(L.OFP_PREC_F32C)
        out.append(ens.forces(L.OFP_PREC_F32C))
    assert torch.equal(*out)
