"""The work that programs built on this library have it do, as cases that can
be timed and whose outputs can be compared.

Every case is one pass through the public entry points (vector_dist.py,
ensemble.py, remote.py and the C ABI's pair passes) on inputs made on the GPU
from a seed:

  sph    a weakly compressible SPH step: ghost_get, updateCellListGPU, Verlet
         rows with a 10 % skin (or the cell walk), density, ghost refresh of
         the density, Tait pressure, force, restoreOrder.  "clustered": the
         periodic cube, half uniform, half in 64 Gaussian clusters.  "column":
         the jittered lattice of a water column, not periodic.
  lj     Lennard-Jones forces, energies and neighbour counts of uniform
         particles in the periodic cube: over the cells, or over a Verlet list
         that getVerletGPU makes anew, as a program does whose particles moved.
  cells  updateCellListGPU with properties carried along, then restoreOrder:
         particles in random order (as generated or loaded), or in cell order
         up to a drift (as a running simulation keeps them).
  boxes  many small periodic LJ boxes as one ensemble: set, a run of velocity
         Verlet steps with its neighbour builds, get.
  run    one large periodic LJ gas from power-law clusters through the same
         engine.
  rank   the one-rank halves of the two exchanges of a decomposed run (cut
         2 x 2 x 2): map (wrap, label, pack) and the remote ghosts (label, pack).

Sizes: 8,192 (the smallest step a program runs at all) to the configured
4,194,304 clustered particles; the LJ boxes 1,024 to 65,536 particles each.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from openfpm_pdata_amd import _lib as L
from openfpm_pdata_amd import ensemble as E
from openfpm_pdata_amd import remote as R
from openfpm_pdata_amd import vector_dist as vdm
from openfpm_pdata_amd import workloads

RHO0, C0, H_COL = workloads.RHO0, workloads.C0, workloads.H_COL
SKIN = 0.10  # SPH and LJ Verlet skin
LJ_NEIGH = 34.3  # neighbours of the uniform LJ gas (65,536 particles, r_c = 0.05)
_TDT = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # the smallest SPH step: a test problem, or the tail of a strong-scaling run; latency
        dict(name="sph_8k", kind="sph", shape="clustered", n=8192, dtype="f32", walk="verlet"),
        # an ordinary step of a study on one GPU, odd size
        dict(name="sph_300k", kind="sph", shape="clustered", n=300007, dtype="f32", walk="verlet"),
        # the configured clustered step, the largest
        dict(name="sph_4m", kind="sph", shape="clustered", n=4194304, dtype="f32", walk="verlet"),
        # the same in plain FP64, for those who want the reference's own precision
        dict(name="sph_f64_400k", kind="sph", shape="clustered", n=400009, dtype="f64", walk="verlet"),
        # a water column without periodic images; the passes walk the cells (no Verlet list kept)
        dict(name="column_1m", kind="sph", shape="column", n=103 ** 3, dtype="f32", walk="cells"),
        # the reference's kind of user loop: FP64 LJ over the 27 cells, 65,536 particles
        dict(name="lj_cells_f64_65k", kind="lj", n=65536, dtype="f64", walk="cells"),
        # one force evaluation after the particles moved: new Verlet list, then the pair pass
        dict(name="lj_verlet_1m", kind="lj", n=1000003, dtype="f32", walk="verlet"),
        # a cell list of particles in the order a file or a generator gives them
        dict(name="cells_random_32m", kind="cells", n=1 << 25, dtype="f32", order="random", per_cell=9.0),
        # a cell list inside a running simulation: last step's order, slightly stale
        dict(name="cells_drifted_5m", kind="cells", n=5000011, dtype="f64", order="drifted", per_cell=9.0),
        # a batch of small molecular-dynamics boxes, sampled together
        dict(name="boxes_64", kind="boxes", n_boxes=64, n_min=1024, n_max=65536, steps=20, precision="f32c"),
        # one large gas, the benchmark's run at an eighth of its particles
        dict(name="run_8m", kind="run", n=1 << 23, steps=40, precision="f32c"),
        # one rank's share of a decomposed clustered run between two steps
        dict(name="rank_4m", kind="rank", n=4194304, dtype="f32"),
    ]


def _log_int(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n | 1 if rng.random() < 0.6 else n


def draw(rng):
    kind = rng.choice(("sph", "sph", "sph", "column", "lj", "lj", "cells", "cells", "boxes", "run", "rank"))
    if kind == "sph":
        if rng.random() < 0.25:
            return dict(kind="sph", shape="clustered", n=_log_int(rng, 8192, 400009), dtype="f64", walk="verlet")
        return dict(kind="sph", shape="clustered", n=_log_int(rng, 8192, 4100000), dtype="f32", walk="verlet")
    if kind == "column":
        return dict(kind="sph", shape="column", n=int(round(math.exp(rng.uniform(math.log(20), math.log(103))))) ** 3,
                    dtype="f32", walk=rng.choice(("cells", "verlet")))
    if kind == "lj":
        if rng.random() < 0.5:
            return dict(kind="lj", n=_log_int(rng, 4096, 262144), dtype=rng.choice(("f64", "f32")), walk="cells")
        return dict(kind="lj", n=_log_int(rng, 16384, 2000000), dtype="f32", walk="verlet")
    if kind == "cells":
        order = rng.choice(("random", "drifted"))
        return dict(kind="cells", n=_log_int(rng, 30000, 30000000), dtype=rng.choice(("f32", "f64")), order=order,
                    per_cell=rng.uniform(3.0, 20.0))
    if kind == "boxes":
        return dict(kind="boxes", n_boxes=rng.randint(8, 64), n_min=1024, n_max=_log_int(rng, 4096, 65536), steps=20,
                    precision=rng.choice(("f32c", "f64")))
    if kind == "run":
        return dict(kind="run", n=_log_int(rng, 1 << 18, 1 << 23), steps=40, precision=rng.choice(("f32c", "f64")))
    return dict(kind="rank", n=_log_int(rng, 65536, 4194304), dtype=rng.choice(("f32", "f64")))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) + 0x0F9D)


def _into(p, dtype):
    """Unit-cube positions in the dtype; values that round up to 1 wrap to 0."""
    p = p.to(dtype)
    return torch.where(p >= 1.0, torch.zeros_like(p), p)


def _uniform(n, seed, dtype):
    return _into(torch.rand((3, n), generator=_gen(seed), device="cuda", dtype=torch.float64), dtype)


def _clustered(n, seed, dtype):
    """workloads.clustered_sph's recipe, made on the GPU."""
    g = _gen(seed)
    nu = n // 2
    nc = n - nu
    uni = torch.rand((3, nu), generator=g, device="cuda", dtype=torch.float64)
    centres = torch.rand((3, 64), generator=g, device="cuda", dtype=torch.float64)
    which = torch.randint(0, 64, (nc,), generator=g, device="cuda")
    clu = centres[:, which] + 0.02 * torch.randn((3, nc), generator=g, device="cuda", dtype=torch.float64)
    return _into(torch.cat([uni, torch.remainder(clu, 1.0)], dim=1), dtype)


def _column(side, seed, dtype):
    """workloads.water_column's recipe, made on the GPU."""
    dx = H_COL / side
    ax = (torch.arange(side, device="cuda", dtype=torch.float64) + 0.5) * dx
    z, y, x = torch.meshgrid(ax, ax, ax, indexing="ij")
    p = torch.stack([x.flatten(), y.flatten(), z.flatten()])
    j = (torch.rand(p.shape, generator=_gen(seed), device="cuda", dtype=torch.float64) * 2.0 - 1.0) * 0.01 * dx
    return (p + j).to(dtype).contiguous()


def _sph_params(case):
    """(box_lo, box_hi, bc, h, mass)"""
    n = case["n"]
    if case["shape"] == "column":
        dx = H_COL / round(n ** (1.0 / 3.0))
        h = 1.3 * dx
        return (-2.0 * h,) * 3, (H_COL + 2.0 * h,) * 3, (0, 0, 0), h, RHO0 * dx ** 3
    return (0.0,) * 3, (1.0,) * 3, (1, 1, 1), 1.3 * n ** (-1.0 / 3.0), RHO0 / n


def _sph_pos(case, seed):
    if case["shape"] == "column":
        return _column(round(case["n"] ** (1.0 / 3.0)), seed, _TDT[case["dtype"]])
    return _clustered(case["n"], seed, _TDT[case["dtype"]])


def _lj_params(case):
    """(r_cut, sigma): a fixed number of neighbours at every size."""
    r = (LJ_NEIGH / (4.0 / 3.0 * math.pi * case["n"])) ** (1.0 / 3.0)
    return r, 0.4 * r


def _box_systems(case, seed):
    """Boxes of log-uniform sizes and r_c ~ U(0.03, 0.08), as workloads.ensemble,
    but on jittered lattices with sigma at most 0.9 of the lattice spacing:
    particles that a run can start from.  Returns (systems, positions, velocities)."""
    rng = np.random.Generator(np.random.PCG64(0x0F9D0004))  # the batch's boxes; the seed moves the particles
    sizes = np.rint(np.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"]), case["n_boxes"]))).astype(int)
    rcs = rng.uniform(0.03, 0.08, case["n_boxes"])
    g = _gen(seed)
    systems, pos = [], []
    for n, rc in zip(sizes, rcs):
        n = int(n)
        m = math.ceil(n ** (1.0 / 3.0) - 1e-9)
        sp = 1.0 / m
        rc = max(float(rc), 1.2 * sp)
        sites = torch.randperm(m ** 3, generator=g, device="cuda")[:n]
        q = torch.stack([sites % m, (sites // m) % m, sites // (m * m)]).double()
        jit = (torch.rand((3, n), generator=g, device="cuda", dtype=torch.float64) - 0.5) * 0.1
        pos.append(_into((q + 0.5 + jit) * sp, torch.float32))
        systems.append(E.System(n, rc, min(0.4 * rc, 0.9 * sp), 1.0, 1.0))
    x = torch.cat(pos, dim=1).contiguous()
    vel = torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float64).float()
    return systems, x, vel


def _box_dt(systems):
    return 2e-3 * min(s.sigma for s in systems)


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"sph": _prepare_sph, "lj": _prepare_lj, "cells": _prepare_cells, "boxes": _prepare_boxes,
            "run": _prepare_run, "rank": _prepare_rank}[case["kind"]](case, seed)


def _prec(dtype):
    return L.OFP_PREC_F32C if dtype == "f32" else L.OFP_PREC_F64


def _prepare_sph(case, seed):
    lo, hi, bc, h, mass = _sph_params(case)
    verlet = case["walk"] == "verlet"
    r = 2.0 * h * (1.0 + SKIN) if verlet else 2.0 * h
    dt = _TDT[case["dtype"]]
    n = case["n"]
    vd = vdm.VectorDistGPU(n, lo, hi, bc, r, dtype=dt, capacity=int(n * (1.0 + 2.2 * r) ** 3) + 2048,
                           props={"rho": (torch.float64, 1), "prs": (torch.float64, 1), "pterm": (dt, 1),
                                  "force": (dt, 3)})
    vd.pos[:, :n] = _sph_pos(case, seed)
    opt = vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION | vdm.CL_QUANT
    sub = 2 if verlet else 1
    cl = vd.getCellListGPU(r / sub, opt, NNIteratorBox=sub, ghostEnlargeFactor=vdm.GHOST_ENLARGE_VL)
    return dict(kind="sph", vd=vd, cl=cl, vl=vdm.VerletListGPU() if verlet else None, r=r, n=n,
                prec=_prec(case["dtype"]), prm=L.SPHParams(h, mass, RHO0, C0))


def _prepare_lj(case, seed):
    r, sigma = _lj_params(case)
    n = case["n"]
    dt = _TDT[case["dtype"]]
    rv = r * (1.0 + SKIN) if case["walk"] == "verlet" else r
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (1, 1, 1), rv, dtype=dt,
                           capacity=int(n * (1.0 + 2.2 * rv) ** 3) + 2048,
                           props={"force": (dt, 3), "energy": (dt, 1), "nn": (torch.int32, 1)})
    vd.pos[:, :n] = _uniform(n, seed, dt)
    cl = None
    if case["walk"] == "cells":
        cl = vd.getCellListGPU(r, vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER_POSITION | vdm.CL_QUANT)
    return dict(kind="lj", vd=vd, cl=cl, r=rv, n=n, prec=_prec(case["dtype"]), prm=L.LJParams(r, sigma, 1.0))


def _prepare_cells(case, seed):
    n, dt = case["n"], _TDT[case["dtype"]]
    r = (case["per_cell"] / n) ** (1.0 / 3.0)
    x = _uniform(n, seed, dt)
    vd = vdm.VectorDistGPU(n, (0.0,) * 3, (1.0,) * 3, (1, 1, 1), r, dtype=dt, capacity=n + 64,
                           props={"id": (torch.int32, 1), "rho": (torch.float64, 1)})
    cl = vd.getCellListGPU(r, vdm.CL_NON_SYMMETRIC | vdm.CL_GPU_REORDER)
    if case["order"] == "drifted":
        # last step's cell order: the list's own cells, then a drift of up to 1 % of a cell per component
        lo = torch.from_numpy(cl.box_lo.astype(np.float64)).cuda()[:, None]
        sp = (torch.from_numpy(cl.box_hi.astype(np.float64)).cuda()[:, None] - lo) / torch.from_numpy(
            cl.div.astype(np.float64)).cuda()[:, None]
        c = torch.floor((x.double() - lo) / sp).long()
        d = torch.from_numpy(cl.div.astype(np.int64)).cuda()
        x = x[:, torch.argsort(c[0] + d[0] * (c[1] + d[1] * c[2]), stable=True)]
        step = (torch.rand(x.shape, generator=_gen(seed + 1), device="cuda", dtype=torch.float64) * 2.0 - 1.0) * 0.01
        x = _into(torch.remainder(x.double() + step * sp, 1.0), dt)
    vd.pos[:, :n] = x
    vd.prp["id"][0, :n] = torch.arange(n, device="cuda", dtype=torch.int32)
    vd.prp["rho"][0, :n] = torch.rand(n, generator=_gen(seed + 2), device="cuda", dtype=torch.float64)
    return dict(kind="cells", vd=vd, cl=cl, n=n)


def _prepare_boxes(case, seed):
    systems, x, vel = _box_systems(case, seed)
    ens = E.Ensemble(systems, torch.float32, E.Options(skin=0.1, sub=2, lanes=8))
    return dict(kind="ens", ens=ens, x=x, vel=vel, dt=_box_dt(systems), steps=case["steps"],
                prec=L.OFP_PREC_F32C if case["precision"] == "f32c" else L.OFP_PREC_F64)


def _prepare_run(case, seed):
    wl, x, vel, _, _ = workloads.power_law_clusters_lj(n=case["n"], seed=workloads.SEED_BASE + 6 + int(seed))
    s = E.System(case["n"], wl.r_cut, wl.params["sigma"], 1.0, 1.0, tuple(wl.box_lo), tuple(wl.box_hi))
    # the options the autotuner picks for this gas
    ens = E.Ensemble([s], torch.float32, E.Options(skin=0.02, sub=1, lanes=1, verlet_rows=2))
    return dict(kind="ens", ens=ens, x=x, vel=vel, dt=wl.params["dt"], steps=case["steps"],
                prec=L.OFP_PREC_F32C if case["precision"] == "f32c" else L.OFP_PREC_F64)


def _prepare_rank(case, seed):
    dt = _TDT[case["dtype"]]
    n_all = case["n"]
    n = n_all // 8
    dims, lo, hi, bc = (2, 2, 2), (0.0,) * 3, (1.0,) * 3, (1, 1, 1)
    r = 2.6 * n_all ** (-1.0 / 3.0) * (1.0 + SKIN)
    slo, shi, sp = R.regular_subdomains(dt, lo, hi, dims)
    _, _, blo, bhi, proc, sid, shifts = R.regular_decomposition(dt, lo, hi, bc, dims, 0, r)
    # rank 0's octant of the clustered particles, moved by up to half the skin since the last map
    half = 0.5 * r * SKIN / (1.0 + SKIN)
    x = 0.5 * _clustered(n, seed, torch.float64)
    x = x + (torch.rand(x.shape, generator=_gen(seed + 1), device="cuda", dtype=torch.float64) * 2.0 - 1.0) * half
    g = _gen(seed + 2)
    n_gho = int(2.0 * n * ((1.0 + 4.4 * r) ** 3 - 1.0)) + 4096
    return dict(kind="rank", x=x.to(dt).contiguous(), n=n, dt=dt,
                f64=torch.rand(n, generator=g, device="cuda", dtype=torch.float64),
                f32=torch.rand(n, generator=g, device="cuda", dtype=torch.float32),
                work=torch.empty((3, n), dtype=dt, device="cuda"), stay=_rank_bufs(n, dt), send=_rank_bufs(n, dt),
                gho=_rank_bufs(n_gho, dt), map=R.Map(dt, slo, shi, sp, np.asarray(lo, slo.dtype),
                                                     np.asarray(hi, slo.dtype), bc, 0),
                ghost=R.GhostRemote(dt, blo, bhi, proc, sid, shifts))


def _rank_bufs(n, dt):
    """A send buffer: positions, an FP64 and an FP32 property."""
    return (torch.zeros((3, n), dtype=dt, device="cuda"), torch.zeros(n, dtype=torch.float64, device="cuda"),
            torch.zeros(n, dtype=torch.float32, device="cuda"))


# --------------------------------------------------------------------- run
def run(state):
    return {"sph": _run_sph, "lj": _run_lj, "cells": _run_cells, "ens": _run_ens, "rank": _run_rank}[
        state["kind"]](state)


def _owned(view, owner):
    """A view of library memory that keeps the handle that owns the memory alive."""
    view.owner = owner
    return view


def _run_sph(s):
    vd, cl, vl, n = s["vd"], s["cl"], s["vl"], s["n"]
    st = vdm._stream()
    vd.ghost_get()
    vd.updateCellListGPU(cl)
    vlh = None
    if vl is not None:
        vl.build(cl, vd.pos, s["r"])
        vlh = vl.h
    rho, prs, pterm, F = (vd.prp[k] for k in ("rho", "prs", "pterm", "force"))
    L.call("ofp_sph_density", cl.h, vlh, vd.pos.data_ptr(), vd.cap, s["prec"], s["prm"], rho.data_ptr(), st)
    vd.ghost_sync_sorted(cl, ("rho",))
    L.call("ofp_sph_eos", s["prec"], rho.data_ptr(), vd.size, s["prm"], prs.data_ptr(), pterm.data_ptr(), st)
    fp = vdm.planes_of(F)
    L.call("ofp_sph_force", cl.h, vlh, vd.pos.data_ptr(), vd.cap, s["prec"], s["prm"], pterm.data_ptr(),
           fp[0][0], fp[1][0], fp[2][0], st)
    vd.restoreOrder(cl, ("force", "rho", "prs"))
    return {"rho": vd.prp["rho"][0, :n], "prs": vd.prp["prs"][0, :n], "force": vd.prp["force"][:, :n]}


def _run_lj(s):
    vd, n = s["vd"], s["n"]
    vd.ghost_get()
    out = {}
    if s["cl"] is not None:
        cl, vlh = vd.updateCellListGPU(s["cl"]), None
    else:
        cl, vl = vd.getVerletGPU(s["r"], vdm.CL_NON_SYMMETRIC | vdm.CL_QUANT, sub=2)
        vlh = vl.h
        out = {"offsets": _owned(vl.arrays()[0], vl)}
    F, U, nn = (vd.prp[k] for k in ("force", "energy", "nn"))
    fp = vdm.planes_of(F)
    L.call("ofp_pair_lj", cl.h, vlh, vd.pos.data_ptr(), vd.cap, s["prec"], s["prm"], fp[0][0], fp[1][0], fp[2][0],
           U.data_ptr(), nn.data_ptr(), vdm._stream())
    vd.restoreOrder(cl, ("force", "energy", "nn"))
    out.update(force=vd.prp["force"][:, :n], energy=vd.prp["energy"][0, :n], nn=vd.prp["nn"][0, :n])
    return out


def _run_cells(s):
    vd, cl, n = s["vd"], s["cl"], s["n"]
    vd.updateCellListGPU(cl, ("id", "rho"))
    # a pass over the sorted particles would run here; then back to the caller's order
    out = dict(sorted_pos=vd.pos[:, :n], sorted_id=vd.prp["id"][0, :n])
    vd.restoreOrder(cl, ("id", "rho"))
    a = cl.arrays()
    out.update(pos=vd.pos[:, :n], id=vd.prp["id"][0, :n], rho=vd.prp["rho"][0, :n], cell_start=a["cell_start"],
               s2n=_owned(a["s2n"], cl), n2s=_owned(a["n2s"], cl))
    return out


def _run_ens(s):
    ens = s["ens"]
    ens.set(s["x"], s["vel"])
    ens.run(s["prec"], s["dt"], s["steps"])
    pos, vel, force = ens.get()
    return {"pos": pos, "vel": vel, "force": force}


def _run_rank(s):
    m, g, n = s["map"], s["ghost"], s["n"]
    x, stay, send, gho = s["work"], s["stay"], s["send"], s["gho"]
    x.copy_(s["x"])  # map wraps in place

    def planes(b):
        return [(b[1].data_ptr(), 8), (b[2].data_ptr(), 4)]

    n_stay, _, _ = m.label(x, n)
    m.pack(x, stay[0], send[0], [(s["f64"].data_ptr(), 8), (s["f32"].data_ptr(), 4)], planes(stay), planes(send))
    # the staying particles' ghosts for the neighbours
    n_out, _ = g.label(stay[0], n_stay)
    if n_out > gho[0].shape[1]:
        gho = s["gho"] = _rank_bufs(n_out, s["dt"])
    g.pack(stay[0], gho[0], planes(stay), planes(gho))
    m_procs, m_counts = m.procs()
    procs, counts = g.procs()
    return {"stay": stay, "send": send, "ghosts": gho, "n_stay": n_stay, "n_send": m.n_send, "n_ghosts": n_out,
            "to": _per_rank(m_procs, m_counts), "ghosts_to": _per_rank(procs, counts)}


def _per_rank(procs, counts):
    """Particles for each of the 8 ranks."""
    out = [0] * 8
    for p, c in zip(procs, counts):
        out[int(p)] = int(c)
    return out


# -------------------------------------------------------------------- work
def _sph_pairs(case):
    """Expected ordered pairs within 2h."""
    n = case["n"]
    v = 4.0 / 3.0 * math.pi * 2.6 ** 3  # neighbours at the mean density
    if case["shape"] == "column":
        return n * v
    own = v / 128.0 / (8.0 * math.pi ** 1.5 * 0.02 ** 3)
    s = (2.6 * n ** (-1.0 / 3.0) / 0.02) ** 2
    own /= (1.0 + 0.15 * s) ** 1.5  # a cut-off that is not small against the cluster
    return n * v + 0.5 * n * own


def work(case):
    """Bytes: positions and properties read once, results written once.  Flops:
    those of the pairs within the cut-off (LJ 23, SPH density 15, force 35)."""
    k = case["kind"]
    s = 8 if case.get("dtype") == "f64" else 4
    if k == "sph":
        n = case["n"]
        return {"bytes": n * (3 * s + 8 + 8 + 3 * s), "flops": 50.0 * _sph_pairs(case)}
    if k == "lj":
        n = case["n"]
        b = n * (3 * s + 4 * s + 4)
        if case["walk"] == "verlet":
            b += n * (8 + 4 * (1.0 + LJ_NEIGH * (1.0 + SKIN) ** 3))
        return {"bytes": b, "flops": 23.0 * n * LJ_NEIGH}
    if k == "cells":
        # sorted copies of positions and both properties, the two permutations, and back
        n = case["n"]
        row = 3 * s + 4 + 8
        return {"bytes": n * (4 * row + 8) + 8 * n / case["per_cell"], "flops": 0}
    if k == "boxes":
        rng = np.random.Generator(np.random.PCG64(0x0F9D0004))
        sizes = np.rint(np.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"]), case["n_boxes"])))
        rcs = np.maximum(rng.uniform(0.03, 0.08, case["n_boxes"]), 1.2 * sizes ** (-1.0 / 3.0))
        pairs = float((sizes * sizes * 4.0 / 3.0 * math.pi * rcs ** 3).sum())
        return {"bytes": float(sizes.sum()) * 60, "flops": 23.0 * pairs * (case["steps"] + 1)}
    if k == "run":
        # about ten neighbours within 2.5 sigma
        return {"bytes": case["n"] * 60, "flops": 23.0 * 10.0 * case["n"] * (case["steps"] + 1)}
    n = case["n"] / 8.0
    return {"bytes": n * 2 * (3 * s + 12) + 0.2 * n * 2 * (3 * s + 12), "flops": 0}


# ------------------------------------------------------------------- exact
_CHUNK = 1 << 25  # candidates expanded at a time


def _pair_sums(x, lo, hi, periodic, r, fn, n_out, per_pair):
    """sum over pairs (i, j), i != j, |x_i - x_j| < r of fn(i, src_j, d, r2), per i:
    (n_out, n) in 64 bits.  x: (3, n) float64."""
    n = x.shape[1]
    lo = torch.tensor(lo, dtype=torch.float64, device="cuda")[:, None]
    hi = torch.tensor(hi, dtype=torch.float64, device="cuda")[:, None]
    parts, src = [x], [torch.arange(n, device="cuda")]
    if periodic:
        w = hi - lo
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    if dx == dy == dz == 0:
                        continue
                    y = x + torch.tensor([[dx], [dy], [dz]], dtype=torch.float64, device="cuda") * w
                    k = ((y > lo - 1.01 * r) & (y < hi + 1.01 * r)).all(dim=0).nonzero().flatten()
                    parts.append(y[:, k])
                    src.append(k)
    p, src = torch.cat(parts, dim=1), torch.cat(src)
    lo2 = torch.minimum(p.min(dim=1, keepdim=True).values, lo) - 1.01 * r
    dims = torch.floor((p.max(dim=1, keepdim=True).values - lo2) / (1.001 * r)).long() + 2
    c = torch.floor((p - lo2) / (1.001 * r)).long()
    key = c[0] + dims[0] * (c[1] + dims[1] * c[2])
    key, order = torch.sort(key)
    p, src = p[:, order], src[order]
    n_cells = int((dims[0] * dims[1] * dims[2]).item())
    start = torch.zeros(n_cells + 1, dtype=torch.long, device="cuda")
    start[1:] = torch.cumsum(torch.bincount(key, minlength=n_cells), 0)
    out = torch.zeros((n_out, n), dtype=torch.float64, device="cuda")
    d0, d1 = int(dims[0]), int(dims[1])
    cell = c[0, :n] + d0 * (c[1, :n] + d1 * c[2, :n])
    by_cell = torch.argsort(cell)  # targets in cell order
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            mid = cell[by_cell] + d0 * (dy + d1 * dz)
            a = start[(mid - 1).clamp(0, n_cells - 1)]
            cnt = start[(mid + 2).clamp(0, n_cells)] - a
            cum = torch.cumsum(cnt, 0)
            total = int(cum[-1].item())
            cuts = torch.searchsorted(cum, torch.arange(_CHUNK, total + _CHUNK, _CHUNK, device="cuda"))
            cuts = [0] + [min(n, int(v) + 1) for v in cuts.tolist()]
            cuts[-1] = n
            for f, e in zip(cuts[:-1], cuts[1:]):
                if e <= f:
                    continue
                t, k = by_cell[f:e], cnt[f:e]
                i = torch.repeat_interleave(t, k)
                base = torch.repeat_interleave(a[f:e] - (torch.cumsum(k, 0) - k), k)
                j = base + torch.arange(i.numel(), device="cuda")
                d = x[:, i] - p[:, j]
                r2 = (d * d).sum(dim=0)
                keep = ((r2 < r * r) & (r2 > 0)).nonzero().flatten()
                if keep.numel():
                    i = i[keep]
                    out.index_add_(1, i, fn(i, src[j[keep]], d[:, keep], r2[keep]))
    return out


def _lj_fn(sigma, eps):
    def fn(i, j, d, r2):
        s6 = (sigma * sigma / r2) ** 3
        return torch.cat([24.0 * eps * (2.0 * s6 * s6 - s6) / r2 * d, (4.0 * eps * (s6 * s6 - s6))[None]])

    return fn


def exact(case, seed):
    k = case["kind"]
    if k == "sph":
        if _sph_pairs(case) > 6e8:
            return None
        lo, hi, bc, h, mass = _sph_params(case)
        x = _sph_pos(case, seed).double()
        a = 1.0 / (math.pi * h ** 3)

        def dens(i, j, d, r2):
            q = torch.sqrt(r2) / h
            w = torch.where(q < 1.0, 1.0 - 1.5 * q * q + 0.75 * q ** 3, 0.25 * (2.0 - q) ** 3)
            return (mass * a * w)[None]

        rho = _pair_sums(x, lo, hi, bool(bc[0]), 2.0 * h, dens, 1, 15)[0] + mass * a
        b = C0 * C0 * RHO0 / 7.0
        prs = b * ((rho / RHO0) ** 7 - 1.0)
        pt = prs / (rho * rho)

        def force(i, j, d, r2):
            rr = torch.sqrt(r2)
            q = rr / h
            dw = a / h * torch.where(q < 1.0, -3.0 * q + 2.25 * q * q, -0.75 * (2.0 - q) ** 2)
            return -mass * (pt[i] + pt[j]) * dw / rr * d

        return {"rho": rho, "prs": prs, "force": _pair_sums(x, lo, hi, bool(bc[0]), 2.0 * h, force, 3, 35)}
    if k == "lj":
        r, sigma = _lj_params(case)
        x = _uniform(case["n"], seed, _TDT[case["dtype"]]).double()
        o = _pair_sums(x, (0.0,) * 3, (1.0,) * 3, True, r, _lj_fn(sigma, 1.0), 4, 23)
        out = {"force": o[:3], "energy": o[3], "nn": None}
        if case["walk"] == "verlet":
            out.update(offsets=None)
        return out
    if k == "boxes":
        w = work(case)
        if w["flops"] / 23.0 > 4e9:
            return None
        systems, x, vel = _box_systems(case, seed)
        dt = _box_dt(systems)
        fs, vs = [], []
        first = 0
        for s in systems:
            p, v = x[:, first:first + s.n].double(), vel[:, first:first + s.n].double()
            first += s.n

            def f():
                q = torch.remainder(p, 1.0)
                return _pair_sums(q, (0.0,) * 3, (1.0,) * 3, True, s.r_cut, _lj_fn(s.sigma, s.eps), 4, 23)[:3]

            F = f()
            for _ in range(case["steps"]):
                v = v + 0.5 * dt * F
                p = p + dt * v
                F = f()
                v = v + 0.5 * dt * F
            fs.append(F)
            vs.append(v)
        # positions are wrapped into the box at neighbour builds only: not compared here
        return {"pos": None, "vel": torch.cat(vs, dim=1), "force": torch.cat(fs, dim=1)}
    return None
