"""A ghost labelling in a captured stream, which it refuses: the handle serves later
calls as if it had not been made."""
import numpy as np
import pytest
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_label_in_a_captured_stream(dtype):
    n = 3000
    x = torch.from_numpy(np.random.default_rng(3).random((3, n))).to(dtype).cuda()
    out = []
    for captured in (False, True):
        vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (1, 1, 1), 0.1, dtype=dtype, capacity=4 * n)
        vd.pos[:, :n] = x
        if captured:
            torch.cuda.synchronize()
            with torch.cuda.graph(torch.cuda.CUDAGraph(), capture_error_mode="relaxed"):
                with pytest.raises(L.OfpError, match="captured"):
                    vd.ghost_get()
        vd.ghost_get()
        out.append(vd.getPosVector().clone())
    assert out[0].shape[1] > n
    assert torch.equal(*out)
