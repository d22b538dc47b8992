"""Device memory that the library keeps of destroyed lists: at most 1/128 of the
device, and given back on request while other handles live."""
import numpy as np
import pytest
import torch

from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


def lists(n, r=0.02):
    x = torch.from_numpy(np.random.default_rng(n).random((3, n))).float().cuda()
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (0, 0, 0), r, dtype=torch.float32)
    vd.pos[:, :n] = x
    return vd.getVerletGPU(r)


def free():
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


def test_trim_gives_everything_back():
    alive = lists(1000)
    vdm.trim()
    f0 = free()
    total = torch.cuda.mem_get_info()[1]
    for n in (200000, 1000000, 3000000, 5000000):  # together more than is kept
        lists(n)
    kept = f0 - free()
    assert 0 < kept <= total // 128 + (64 << 20)
    assert vdm.trim() > 0
    assert f0 - free() <= 64 << 20  # what the runtime itself holds
    assert vdm.trim() == 0
    off, _ = alive[1].arrays()
    assert int(off[0]) == 0
    lists(200000)  # and lists are made as before
