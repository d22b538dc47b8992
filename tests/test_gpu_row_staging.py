"""One Verlet row per lane against 16 lanes per row at the row lengths where a wave's
staged entries end (1532 of 64 rows): jittered lattices with 7 to 93 entries a row,
in boxes whose waves are full, partial, and of two systems.  Neighbour counts exact,
forces to the rounding of their FP32 storage (the partial sums' order differs)."""
import numpy as np
import pytest

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import ensemble as E
from test_gpu_tiles import _forces_nn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shell", [1.1, 1.5, 1.55, 1.8, 2.1, 2.3])
@pytest.mark.parametrize("m", [(9,), (10, 7), (13,)])
def test_lanes_agree(m, shell):
    rng = np.random.default_rng(7)
    systems, pos = [], []
    for k in m:
        q = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij")).reshape(3, -1) + 0.5
        q = q[:, rng.permutation(k ** 3)] + (rng.random((3, k ** 3)) - 0.5) * 0.05
        systems.append(E.System(k ** 3, shell / k, 0.9 / k, 1.0, 1.0))
        pos.append((q / k).astype(np.float32))
    a = _forces_nn(systems, pos, E.Options(skin=0.05, sub=1, lanes=1))
    b = _forces_nn(systems, pos, E.Options(skin=0.05, sub=1, lanes=16))
    for prec in (L.OFP_PREC_F64, L.OFP_PREC_F32C):
        np.testing.assert_array_equal(a[prec][2], b[prec][2])
        # either side rounds a force to FP32 once: 2^-24 of the largest component each
        scale = np.abs(b[prec][0]).max()
        assert np.abs(a[prec][0] - b[prec][0]).max() <= 2.0 ** -22 * scale
