"""An ensemble that is given particles, computes forces and runs, more than once:
its captured graphs name the buffers of earlier runs.  Replays equal direct launches
bit for bit, in positions, velocities and forces."""
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import ensemble as E
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


def gas(systems, m, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    pos, vel = [], []
    for s in systems:
        c = torch.randperm(m ** 3, generator=g, device="cuda")[: s.n]
        q = torch.stack([c % m, (c // m) % m, c // (m * m)]).double() + 0.5
        q = q + (torch.rand(q.shape, generator=g, device="cuda", dtype=torch.float64) - 0.5) * 0.1
        pos.append((q / m).float())
        vel.append(torch.randn((3, s.n), generator=g, device="cuda", dtype=torch.float64).float())
    return torch.cat(pos, dim=1).contiguous(), torch.cat(vel, dim=1).contiguous()


@pytest.mark.parametrize("explicit", [False, True])
@pytest.mark.parametrize("steps", [1, 2, 3])
@pytest.mark.parametrize("prec", [L.OFP_PREC_F64, L.OFP_PREC_F32C])
def test_set_forces_run_again(prec, steps, explicit):
    """Each run starts with a rebuild; explicit: a rebuild by hand stands before it."""
    m = 14
    systems = [E.System(m ** 3, 0.16, 0.8 / m, 1.0, 1.0), E.System(1500, 0.16, 0.8 / m, 1.0, 1.0)]
    ens = [E.Ensemble(systems, torch.float32, E.Options(skin=0.1, sub=1, lanes=1, headroom=1.5)) for _ in range(2)]
    for rnd in range(4):
        x, v = gas(systems, m, rnd)
        for again in range(2):  # the second time without set
            out = []
            for e, graph in zip(ens, (False, True)):
                if again == 0:
                    e.set(x, v)
                    e.force_pass(prec)
                if explicit:
                    e.rebuild(sizing=False)
                e.test_masks(0, pending=True)
                e.run(prec, 1e-4, steps, use_graph=graph)
                out.append(e.get())
            for name, a, b in zip(("pos", "vel", "force"), *out):
                assert torch.equal(a, b), (rnd, again, name)


@pytest.mark.parametrize("with_forces", [False, True])
@pytest.mark.parametrize("n", [2000, 1 << 22])
def test_arrays_of_a_run_without_rebuild(n, with_forces):
    """A run that needs no rebuild reorders the stored particles but moves no buffer."""
    m = round(n ** (1.0 / 3.0)) + 1
    systems = [E.System(n, 1.5 / m, 0.5 / m, 1.0, 1.0)]
    ens = E.Ensemble(systems, torch.float32, E.Options(skin=0.3, sub=1, lanes=1))
    x, v = gas(systems, m, 1)
    ens.set(x, v)
    if with_forces:
        ens.force_pass(L.OFP_PREC_F64)
    else:
        ens.rebuild()
    a = ens.arrays()
    before = ens.status()["rebuilds"]
    ens.run(L.OFP_PREC_F64, 1e-6 / m, 3)
    assert ens.status()["rebuilds"] == before
    b = ens.arrays()
    assert (a.pos, a.vel, a.force, a.gid, a.cap) == (b.pos, b.vel, b.force, b.gid, b.cap)
    gid = ens.gid().long()
    assert torch.equal(torch.sort(gid).values, torch.arange(n, device="cuda"))
    for ptr, want in zip((a.pos, a.vel, a.force), ens.get()):
        got = vdm.device_view(ptr, 3 * int(a.cap), torch.float32).view(3, -1)[:, :n]
        assert torch.equal(got, want[:, gid])


@pytest.mark.parametrize("n", [2000, (1 << 22) + 3])
def test_positions_changed_by_their_pointer(n):
    """Particles that the caller moves after a build, by more than the skin allows: the
    next run rebuilds, in three steps at once as in three runs of one step."""
    m = round(n ** (1.0 / 3.0)) + 1
    systems = [E.System(n, 1.5 / m, 0.5 / m, 1.0, 1.0)]
    x, v = gas(systems, m, 4)
    out = []
    for split in (False, True):
        ens = E.Ensemble(systems, torch.float32, E.Options(skin=0.1, sub=1, lanes=1))
        ens.set(x, v)
        ens.rebuild()
        a = ens.arrays()
        pos = vdm.device_view(a.pos, 3 * int(a.cap), torch.float32).view(3, -1)
        pos[0, :n:5] += 0.6 / m
        before = ens.status()["rebuilds"]
        for _ in range(3 if split else 1):
            ens.run(L.OFP_PREC_F64, 1e-7 / m, 1 if split else 3)
        assert ens.status()["rebuilds"] == before + 1
        out.append(ens.get())
        del ens
    for a, b in zip(*out):
        assert torch.equal(a, b)
