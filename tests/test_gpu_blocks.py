"""Device blocks pass from destroyed lists to new ones: lists made and dropped
one after another, on several streams and from several threads, are those of
lists that stay."""
import threading

import numpy as np
import pytest
import torch

from openfpm_pdata_amd import vector_dist as vdm

pytestmark = pytest.mark.gpu


def particles(n, seed):
    return torch.from_numpy(np.random.default_rng(seed).random((3, n))).float().cuda()


def make(x, r=0.06):
    n = x.shape[1]
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (1, 1, 1), r, dtype=torch.float32, capacity=2 * n + 64)
    vd.pos[:, :n] = x
    vd.ghost_get()
    cl, vl = vd.getVerletGPU(r)
    return vd, cl, vl


def entries(made):
    off, nbr = made[2].arrays()
    return off.clone(), nbr.clone()


def test_lists_made_anew_equal_lists_that_stay():
    sizes = (3000, 20000, 3100, 50000, 2900)
    kept = [make(particles(n, k)) for k, n in enumerate(sizes)]  # blocks of their own
    want = [entries(m) for m in kept]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for rnd in range(4):
        for k, n in enumerate(sizes):
            with torch.cuda.stream(streams[(rnd + k) % 2]):
                m = make(particles(n, k))
                got = entries(m)
                del m  # its kernels and copies may still run; the next list takes its blocks
            for a, b in zip(got, want[k]):
                torch.cuda.current_stream().wait_stream(streams[(rnd + k) % 2])
                assert torch.equal(a, b)
    del kept


def test_threads():
    want = [entries(make(particles(8000 + 500 * t, 50 + t))) for t in range(4)]
    torch.cuda.synchronize()
    bad = []

    def work(t):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(6):
                    m = make(particles(8000 + 500 * t, 50 + t))
                    got = entries(m)
                    del m
                    if not all(torch.equal(a, b) for a, b in zip(got, want[t])):
                        bad.append(t)
        except Exception as e:  # noqa: BLE001
            bad.append((t, repr(e)))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_kept_blocks_are_bounded():
    free0, total = torch.cuda.mem_get_info()
    for k in range(12):
        make(particles(1000 * (k + 1) ** 2, k), 0.03)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free1, _ = torch.cuda.mem_get_info()
    assert free0 - free1 <= total // 32 + (1 << 28)
