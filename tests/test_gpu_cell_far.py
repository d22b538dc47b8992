"""Permutations far from cell order (restore, reorder, the build's own planes), which
go by ranges of destinations from 2^22 particles: against the plain gather and
scatter in torch, exact, at the edges of tiles and ranges and for planes of both
element sizes in orders that leave them unaligned to one another in the scratch."""
import pytest
import torch

from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


def _planes(n, sizes, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = {4: torch.int32, 8: torch.int64}
    return [torch.randint(-2**31, 2**31 - 1, (n,), generator=gen, device="cuda").to(dt[b]) for b in sizes]


def _args(planes):
    return [(p.data_ptr(), p.element_size()) for p in planes]


@pytest.mark.parametrize("order", ["random", "near", "exact"])
@pytest.mark.parametrize("n", [(1 << 22) - 1, 1 << 22, (1 << 22) + 1, (1 << 22) + 32767, (1 << 23) - 1, (1 << 25) + 5])
def test_far(n, order):
    side = 64
    gen = torch.Generator(device="cuda").manual_seed(n)
    pos = torch.rand((3, n), generator=gen, device="cuda") * side

    def cells(p):
        c = torch.clamp(torch.floor(p).long() + 1, max=side + 1)
        return c[0] + (side + 2) * (c[1] + (side + 2) * c[2])

    if order != "random":
        pos = pos[:, torch.argsort(cells(pos), stable=True)].contiguous()
        if order == "near":
            pos[:, [0, n - 2]] = pos[:, [n - 2, 0]]
    perm = torch.argsort(cells(pos), stable=True)
    sizes = [4, 8, 4, 4, 8, 8, 4]
    src = _planes(n, sizes, n + 1)
    for with_pos in (True, False):
        opt = vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_PROPERTY
        opt |= vdm.CL_GPU_REORDER_POSITION if with_pos else 0
        cl = vdm.CellListGPU(torch.float32, (0.0,) * 3, (float(side),) * 3, (side,) * 3, opt, 1.0)
        out = torch.empty_like(pos) if with_pos else None
        dst = [torch.zeros_like(p) for p in src]
        cl.construct(pos, n, n, out, _args(src), _args(dst))
        assert torch.equal(cl.arrays()["s2n"].long(), perm)
        assert torch.equal(cl.arrays()["n2s"].long()[perm], torch.arange(n, device="cuda"))
        for a, b in zip(src, dst):
            assert torch.equal(b, a[perm])
        back = [torch.zeros_like(p) for p in src]
        cl.restore(_args(dst), _args(back))
        for a, b in zip(src, back):
            assert torch.equal(a, b)
        again = [torch.zeros_like(p) for p in src]
        cl.reorder(_args(src), _args(again))
        for a, b in zip(dst, again):
            assert torch.equal(a, b)


@pytest.mark.parametrize("n", [3072 << 15, (3072 << 15) + 1])
def test_far_most_particles(n):
    """The most ranges (3072), and one particle more (the direct kernels again)."""
    side = 200
    pos = torch.rand((3, n), generator=torch.Generator(device="cuda").manual_seed(9), device="cuda") * side
    cl = vdm.CellListGPU(torch.float32, (0.0,) * 3, (float(side),) * 3, (side,) * 3,
                         vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER, 1.0)
    src = _planes(n, [4, 8], 11)
    dst = [torch.zeros_like(p) for p in src]
    out = torch.empty_like(pos)
    cl.construct(pos, n, n, out, _args(src), _args(dst))
    s2n = cl.arrays()["s2n"].long()
    assert torch.equal(cl.arrays()["n2s"].long()[s2n], torch.arange(n, device="cuda"))
    assert torch.equal(out, pos[:, s2n])
    for a, b in zip(src, dst):
        assert torch.equal(b, a[s2n])
    back = [torch.zeros_like(p) for p in src]
    cl.restore(_args(dst), _args(back))
    for a, b in zip(src, back):
        assert torch.equal(a, b)


def test_far_most_planes():
    """24 planes, the most a call takes, with the positions (3 more)."""
    n, side = (1 << 22) + 11, 64
    pos = torch.rand((3, n), generator=torch.Generator(device="cuda").manual_seed(5), device="cuda") * side
    cl = vdm.CellListGPU(torch.float32, (0.0,) * 3, (float(side),) * 3, (side,) * 3,
                         vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER, 1.0)
    src = _planes(n, [4, 8, 4] * 8, 7)
    dst = [torch.zeros_like(p) for p in src]
    out = torch.empty_like(pos)
    cl.construct(pos, n, n, out, _args(src), _args(dst))
    s2n = cl.arrays()["s2n"].long()
    assert torch.equal(out, pos[:, s2n])
    for a, b in zip(src, dst):
        assert torch.equal(b, a[s2n])


def test_far_streams():
    """Restores of one list on two streams share its scratch one after another."""
    n, side = (1 << 22) + 3, 64
    pos = torch.rand((3, n), generator=torch.Generator(device="cuda").manual_seed(3), device="cuda") * side
    cl = vdm.CellListGPU(torch.float32, (0.0,) * 3, (float(side),) * 3, (side,) * 3,
                         vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION, 1.0)
    out = torch.empty_like(pos)
    cl.construct(pos, n, n, out)
    s2n = cl.arrays()["s2n"].long()
    src = [_planes(n, [4, 8], k) for k in range(4)]
    dst = [[torch.zeros_like(p) for p in s] for s in src]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for k in range(4):
        with torch.cuda.stream(streams[k % 2]):
            cl.restore(_args(src[k]), _args(dst[k]))
    torch.cuda.synchronize()
    for k in range(4):
        for a, b in zip(src[k], dst[k]):
            assert torch.equal(b[s2n], a)
