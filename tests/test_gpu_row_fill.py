"""The thread-per-row list fill at the rows' lengths where its staging ends (1024 and
2560 entries of 64 rows) and past it: clumps of m particles far from one another,
so every row is its clump, in ascending sorted order."""
import numpy as np
import pytest
import torch

from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("sub", [1, 2, 3])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 39, 40, 41, 70])
def test_rows(m, sub, dtype):
    rng = np.random.default_rng(m)
    g = 5
    c = (np.stack(np.meshgrid(*[np.arange(g)] * 3, indexing="ij")).reshape(3, -1) + 0.5) / g
    pos = c[:, :, None] + (rng.random((3, g ** 3, m)) - 0.5) * 0.008
    n = pos[0].size
    r = 0.02
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (0, 0, 0), r, dtype=dtype)
    vd.pos[:, :n] = torch.from_numpy(pos.reshape(3, n)).to(dtype).cuda()
    cl, vl = vd.getVerletGPU(r, vdm.CL_NON_SYMMETRIC, sub=sub)
    off, nbr = vl.arrays()
    assert torch.equal(off.long(), torch.arange(n + 1, device="cuda") * m)
    s2n = cl.arrays()["s2n"].long()[:n]
    dom = cl.arrays()["dom"].long()[:n]
    rows = nbr[: n * m].long().view(n, m)
    assert bool((rows[:, 1:] > rows[:, :-1]).all())
    assert torch.equal(s2n[rows] // m, (s2n[dom] // m)[:, None].expand(n, m))
