"""Runs of many particles given in random order: the reordering into cell order and
the way back go by ranges of destinations (from 2^22 particles).  A run of three
steps equals three runs of one step, which keep the caller's order, bit for bit."""
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import ensemble as E
from test_gpu_run_order import shuffled_lattices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [(1 << 22) + 1, 162 ** 3])
def test_far_run_equals_single_steps(n, dtype):
    systems, x, v = shuffled_lattices((n,))
    systems = [E.System(n, 1.6 / 162, 0.8 / 162, 1.0, 1.0)]
    x, v = x.to(dtype).cuda(), v.to(dtype).cuda()
    out = []
    for split in (False, True):
        ens = E.Ensemble(systems, dtype, E.Options(skin=0.1, sub=1, lanes=1))
        ens.set(x, v)
        for _ in range(3 if split else 1):
            ens.run(L.OFP_PREC_F32C, 1e-7, 1 if split else 3)
        out.append(ens.get())
        only = ens.get()[1]
        assert torch.equal(only, out[-1][1])
        del ens
    for a, b in zip(*out):
        assert torch.equal(a, b)
    assert not torch.equal(out[0][0], x)
