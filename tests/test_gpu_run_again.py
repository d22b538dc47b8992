"""An ensemble that is given particles, computes forces and runs, more than once:
its captured graphs name the buffers of earlier runs.  Replays equal direct launches
bit for bit, in positions, velocities and forces."""
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import ensemble as E

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
