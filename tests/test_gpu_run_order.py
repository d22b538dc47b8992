"""A run whose particles are still in the caller's order puts them in cell order
before its steps (ofp_ens_run of two or more steps).  The sorted order, the
lists and the arithmetic stay, so a run of n steps equals n runs of one step,
which keep the caller's order, bit for bit; neighbour builds that follow read
the new order."""
import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import ensemble as E
from openfpm_pdata_amd.vector_dist import device_view

pytestmark = pytest.mark.gpu


def shuffled_lattices(sizes, seed=5):
    rng = np.random.default_rng(seed)
    systems, pos, vel = [], [], []
    for n in sizes:
        m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
        s = rng.permutation(m ** 3)[:n]
        q = np.stack([s % m, (s // m) % m, s // (m * m)]) + 0.5 + (rng.random((3, n)) - 0.5) * 0.1
        rc = max(0.12, 2.2 / m) if m > 4 else 0.2
        systems.append(E.System(n, rc, 0.8 / m if m > 1 else 0.05, 1.0, 1.0))
        pos.append((q / m).astype(np.float32))
        vel.append(rng.standard_normal((3, n)).astype(np.float32))
    return systems, torch.from_numpy(np.concatenate(pos, axis=1)), torch.from_numpy(np.concatenate(vel, axis=1))


@pytest.mark.parametrize("walk", [0, 1])
@pytest.mark.parametrize("prec", [L.OFP_PREC_F64, L.OFP_PREC_F32C])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("sizes", [(1,), (257,), (4913,), (1000, 1, 63, 2744)])
def test_run_equals_single_steps(sizes, dtype, prec, walk):
    systems, x, v = shuffled_lattices(sizes)
    x, v = x.to(dtype).cuda(), v.to(dtype).cuda()
    opts = E.Options(skin=0.1, sub=1, lanes=1, pair_walk=walk)
    out = []
    for split in (False, True):
        ens = E.Ensemble(systems, dtype, opts)
        ens.set(x, v)
        if split:
            for _ in range(5):
                ens.run(prec, 1e-5, 1)
        else:
            ens.run(prec, 1e-5, 5)
        out.append(ens.get())
        assert ens.status()["rebuilds"] == 1
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_relabelled_storage_is_consistent():
    """After the reordering: gid is the permutation of the stored particles, the
    sorted slots name the new storage indices, and a later rebuild gives the same
    forces (the ghosts' sources: the bit-equality above)."""
    systems, x, v = shuffled_lattices((3375, 700))
    x, v = x.cuda(), v.cuda()
    ens = E.Ensemble(systems, torch.float32, E.Options(skin=0.1, sub=2, lanes=8))
    ens.set(x, v)
    ens.run(L.OFP_PREC_F64, 0.0, 3)  # dt 0: the configuration stays
    gid = ens.gid().long()
    assert torch.equal(torch.sort(gid).values, torch.arange(ens.N, device="cuda"))
    a = ens.arrays()
    P = device_view(a.pos, 3 * int(a.cap), torch.float32).view(3, -1)
    assert torch.equal(P[:, : ens.N], x[:, gid])
    cv, _ = ens.lists()
    n = ens.N + int(ens.status()["n_ghost"])
    s2n = device_view(cv.sort_to_nonsort, n, torch.int32).long()
    n2s = device_view(cv.nonsort_to_sort, n, torch.int32).long()
    dom = device_view(cv.dom_sort_ids, ens.N, torch.int32).long()
    assert torch.equal(s2n[n2s], torch.arange(n, device="cuda"))
    assert torch.equal(s2n[dom], torch.arange(ens.N, device="cuda"))
    f0 = ens.get()[2]
    ens.rebuild(sizing=False)
    f1 = ens.forces(L.OFP_PREC_F64)
    # the same pairs; ghosts may come in another order inside a cell: rounding of the sums only
    assert float((f0 - f1).abs().max()) <= 1e-5 * float(f0.abs().max())
