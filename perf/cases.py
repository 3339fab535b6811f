"""The work that programs have this framework do, as cases that can be timed.

What a user calls: the pressure solve of one mesh (device arrays, or host arrays through the plugin factory), the
pressure step around it, the solve of a batch of meshes, the operators of the time step either side of the solve, a
whole time step of the flow past a disk, and a mesh change.  Sizes are those of ``cup2d_amd.workloads`` (128 blocks,
1448, about 8.3k and 16k, the 64-instance batch) and ragged ones between.

The solves' right-hand sides are b = A x for a smooth mean-free x made from the seed, so that x is the exact answer;
they are solved to a relative residual of 1e-12, as where pressures are compared with the CPU's.  Vectors live in
torch tensors whose addresses are handed to the solver.
"""

import functools
import math
from types import SimpleNamespace

import numpy as np
import torch

from cup2d_amd import flow as F
from cup2d_amd import mesh as M
from cup2d_amd import poisson as PS
from cup2d_amd import workloads as W

TOL = 1e-12
TOL_INF = 1e-13  # in the infinity norm, which bounds the smooth part of the error less tightly
STEP_TOL = 1e-11  # the step's mixed solver stops on the recomputed residual, whose rounding floor there is 2e-12
MIXED_MOST = 3000  # blocks up to which that floor lies below TOL
MAX_ITER = 12000


class Vec:
    """A device vector held by torch, as the solver's methods take it."""

    def __init__(self, t):
        self.t, self.ptr, self.n = t, t.data_ptr(), t.numel()


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest solve: 16 x 8 uniform blocks, one call per time step of a small run
        dict(name="solve 128 blocks", kind="solve", mesh="uniform", bx=16, by=8, px=False, py=False, precision="fp64",
             norm="l2", mean=0),
        # an odd grid, periodic in x, in the stopping norm of the GPU solver being replaced
        dict(name="solve 37x23 periodic", kind="solve", mesh="uniform", bx=37, by=23, px=True, py=False,
             precision="fp64", norm="inf", mean=0),
        # the plugin boundary: makePoissonSolver(...).solve(input, output) on host arrays, 3 levels around a disk
        dict(name="plugin 1448 blocks", kind="plugin", mesh="graded", precision="fp64"),
        # the same mesh, mixed precision, device arrays
        dict(name="mixed 1448 blocks", kind="solve", mesh="graded", precision="mixed", norm="l2", mean=0),
        # the mean-row form of the operator (bMeanConstraint)
        dict(name="mean row 104 blocks", kind="solve", mesh="disks", seed=7, levels=3, target=104, precision="fp64",
             norm="l2", mean=1),
        # the pressure step of the cylinder flow's static mesh: rhs - L p_old, the solve, the mean
        dict(name="pressure step 8k blocks", kind="pstep", mesh="cylinder", precision="fp64"),
        # the largest single mesh: 6 levels around 4 disks, 1.04M unknowns
        dict(name="solve 16k blocks 6 levels", kind="solve", mesh="amr6", precision="fp64", norm="l2", mean=0),
        # many independent meshes in one call, 512 to 8192 blocks each: the measured batch
        dict(name="batch 64", kind="batch", seed=4, count=64, nmin=512, nmax=8192, precision="fp64"),
        # a small ensemble in mixed precision
        dict(name="batch 9 mixed", kind="batch", seed=11, count=9, nmin=300, nmax=3000, precision="mixed"),
        # the operators before and after the solve on a large uniform grid: advection-diffusion, divergence, correction
        dict(name="operators 1M cells", kind="operators", bx=128, by=128, px=False, py=False),
        # a whole time step of the flow past the cylinder (static mesh, mixed precision)
        dict(name="time step 8k blocks", kind="step", levels=5, target=8192, precision="mixed"),
        # a mesh change: score, new tree, fields carried over, operator assembled, on the 6-level mesh
        dict(name="mesh change 16k blocks", kind="adapt", mesh="amr6"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solve", "solve", "solve", "disks", "disks", "plugin", "pstep", "batch", "batch", "operators",
                       "adapt"])
    precision = rng.choice(["fp64", "fp64", "mixed"])
    norm = rng.choice(["l2", "inf"])
    if kind == "solve":
        mean = 1 if rng.random() < 0.2 else 0
        top = 256 if mean else MIXED_MOST if precision == "mixed" else 6000
        nb = log(30, top)
        bx = max(1, log(math.sqrt(nb) / 2, math.sqrt(nb) * 2))
        by = max(1, min(nb // bx, 8 * bx))
        px, py = (False, False) if mean else (rng.random() < 0.3, rng.random() < 0.3)
        # a periodic direction has at least 3 blocks
        return dict(kind="solve", mesh="uniform", bx=max(bx, 3), by=max(by, 3), px=px, py=py, precision=precision,
                    norm=norm if precision == "fp64" else "l2", mean=mean)
    seed, levels = rng.randrange(1 << 20), rng.randint(2, 5)
    # every level more than two starts from 128 blocks at level 0 (levels - 1 refinements)
    target = log(260, 1200 if levels < 4 else 12000 if precision == "fp64" or kind == "adapt" else MIXED_MOST)
    if kind == "disks":
        return dict(kind="solve", mesh="disks", seed=seed, levels=levels, target=target, precision=precision, norm="l2",
                    mean=0)
    if kind == "plugin":
        return dict(kind="plugin", mesh="disks", seed=seed, levels=min(levels, 3), target=min(target, 1200),
                    precision=precision)
    if kind == "pstep":
        return dict(kind="pstep", mesh="disks", seed=seed, levels=levels, target=target, precision=precision)
    if kind == "batch":
        lo = log(260, 1000)
        hi = lo * rng.randint(1, 8)
        return dict(kind="batch", seed=seed, count=log(2, 32), nmin=lo,
                    nmax=max(lo, min(hi, MIXED_MOST)) if precision == "mixed" else hi, precision=precision)
    if kind == "operators":
        return dict(kind="operators", bx=log(3, 150), by=log(3, 120), px=rng.random() < 0.4, py=rng.random() < 0.4)
    return dict(kind="adapt", mesh="disks", seed=seed, levels=levels, target=target)


# ---------------------------------------------------------------------------
# meshes and operators (made once: a program keeps its mesh)
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _make_mesh(what, *a):
    if what == "uniform":
        bx, by, px, py = a
        return M.uniform(bx, by, extent=max(bx, by) / 8.0, periodic_x=px, periodic_y=py)
    if what == "disks":
        seed, levels, target = a
        rng = np.random.default_rng(seed)
        disks = [(float(rng.uniform(0.3, 1.7)), float(rng.uniform(0.25, 0.75)), float(rng.uniform(0.05, 0.15)))]
        return W._bisect_mesh(lambda s: M.graded(16, 8, levels, 2.0, disks, [s * 0.4 * 0.5**k for k in range(levels - 1)]),
                              target, 0.05)
    if what == "cylinder":
        return W.cylinder_mesh(*a)
    return {"graded": W.graded_disk_mesh, "amr6": W.four_disk_amr6_mesh}[what]()


def _mesh(case):
    what = case["mesh"]
    if what == "uniform":
        return _make_mesh(what, case["bx"], case["by"], case["px"], case["py"])
    if what == "disks":
        return _make_mesh(what, case["seed"], case["levels"], case["target"])
    return _make_mesh(what)


@functools.lru_cache(maxsize=None)
def _make_batch(seed, count, nmin, nmax):
    if (seed, count, nmin, nmax) == (4, 64, 512, 8192):
        return W.batch64_meshes()
    return W.batch64_meshes(seed, count, nmin, nmax)


def _batch(case):
    return _make_batch(case["seed"], case["count"], case["nmin"], case["nmax"])


def _kept(m, key, make):
    """Kept with the mesh, which lives as long as this module."""
    if key not in m.meta:
        m.meta[key] = make()
    return m.meta[key]


def _operator(meshes):
    """The meshes' block-diagonal operator: (col, val) of the rows' first 5 entries, and (row, col, val) of the rest."""
    return _kept(meshes[0], "operator of %d" % len(meshes), lambda: _assemble(meshes))


def _assemble(meshes):
    parts, rest, off = [], [], 0
    for m in meshes:
        rp, col, val, _ = PS.assemble_csr(m, 0)
        n = m.n
        c, v = np.zeros((5, n), np.int64), np.zeros((5, n))
        length = np.diff(rp)
        for k in range(5):
            has = length > k
            c[k, has], v[k, has] = col[rp[:-1][has] + k], val[rp[:-1][has] + k]
        long_ = np.nonzero(length > 5)[0]
        if long_.size:
            width = int(length.max()) - 5
            lc, lv = np.zeros((width, long_.size), np.int64), np.zeros((width, long_.size))
            for k in range(width):
                has = length[long_] > k + 5
                at = rp[:-1][long_[has]] + k + 5
                lc[k, has], lv[k, has] = col[at], val[at]
            rest.append((long_ + off, lc + off, lv))
        parts.append((c + off, v))
        off += n
    cols = torch.from_numpy(np.concatenate([p[0] for p in parts], axis=1).astype(np.int32)).cuda()
    vals = torch.from_numpy(np.concatenate([p[1] for p in parts], axis=1)).cuda()
    extra = [tuple(torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in r) for r in rest]
    return cols, vals, extra


def _apply(meshes, x):
    cols, vals, extra = _operator(meshes)
    y = torch.zeros_like(x)
    for k in range(5):
        y += vals[k] * x[cols[k].long()]
    for row, c, v in extra:
        for k in range(c.shape[0]):
            y[row] += v[k] * x[c[k]]
    return y


def _cells(m):
    return _kept(m, "cells", lambda: tuple(torch.from_numpy(a).cuda()
                                           for a in (*m.cell_centers(), np.repeat(m.h2(), 64))))


def _pressure(m, seed):
    """A smooth mean-free pressure: 16 Gaussian bumps of either sign and of the sizes of vortices and bodies."""
    x, y, h2 = _cells(m)
    rng = np.random.default_rng(seed)
    lx, ly = m.domain()
    p = torch.zeros_like(x)
    for _ in range(16):
        cx, cy, s, a = rng.uniform(0, lx), rng.uniform(0, ly), rng.uniform(0.04, 0.3), rng.normal()
        dx, dy = x - cx, y - cy
        if m.periodic_x:
            dx = dx - lx * torch.round(dx / lx)
        if m.periodic_y:
            dy = dy - ly * torch.round(dy / ly)
        p += a * torch.exp(-(dx * dx + dy * dy) / (2 * s * s))
    return p - (p * h2).sum() / h2.sum()


def _velocity(m, seed):
    """Two velocity components of a few vortices (periodic directions: of their lattice)."""
    x, y, _ = _cells(m)
    rng = np.random.default_rng(seed)
    lx, ly = m.domain()
    u, v = torch.zeros_like(x), torch.zeros_like(x)
    for _ in range(6):
        kx, ky = int(rng.integers(1, 4)), int(rng.integers(1, 4))
        a, f = 0.1 * rng.normal(), rng.uniform(0, 2 * math.pi, 2)
        sx, sy = 2 * math.pi * kx / lx * x + f[0], 2 * math.pi * ky / ly * y + f[1]
        u += a * (2 * math.pi * ky / ly) * torch.sin(sx) * torch.cos(sy) / 10
        v -= a * (2 * math.pi * kx / lx) * torch.cos(sx) * torch.sin(sy) / 10
    return u, v


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------

def _config(case):
    return dict(precision=PS.MIXED if case["precision"] == "mixed" else PS.FP64,
                norm=PS.NORM_INF if case.get("norm") == "inf" else PS.NORM_L2, max_iter=MAX_ITER)


def prepare(case, seed):
    return {"solve": _prepare_solve, "plugin": _prepare_plugin, "pstep": _prepare_pstep, "batch": _prepare_batch,
            "operators": _prepare_operators, "step": _prepare_step, "adapt": _prepare_adapt}[case["kind"]](case, seed)


def run(state):
    return state.run(state)


def _prepare_solve(case, seed):
    m = _mesh(case)
    b = _apply((m,), _pressure(m, seed))
    s = PS.Solver(mean_constraint=case["mean"], **_config(case)).set_mesh(m, on_device=True)
    return SimpleNamespace(s=s, b=Vec(b), x=Vec(torch.zeros_like(b)), run=_run_solve,
                           tol=TOL_INF if case["norm"] == "inf" else TOL)


def _run_solve(st):
    st.x.t.zero_()  # the initial guess
    torch.cuda.current_stream().synchronize()  # the solver has a stream of its own
    st.s.solve_device(st.b, st.x, rel_tol=st.tol)
    return st.x.t


def _prepare_plugin(case, seed):
    m = _mesh(case)
    b = _apply((m,), _pressure(m, seed)).cpu().numpy()
    sim = PS.SimulationData(poissonSolver="hip_mixed" if case["precision"] == "mixed" else "cuda_iterative",
                            PoissonTol=0.0, PoissonTolRel=TOL_INF if case["precision"] == "fp64" else TOL, maxPoissonRestarts=100, maxPoissonIterations=MAX_ITER,
                            step=20)
    sim.tmp, sim.pres = PS.ScalarGrid(m, b.reshape(-1, 8, 8)), PS.ScalarGrid(m)
    solver = PS.makePoissonSolver(sim)
    solver.solver.set_mesh(m, on_device=True)
    solver._mesh, sim.pres.UpdateFluxCorrection = m, False
    return SimpleNamespace(sim=sim, solver=solver, run=_run_plugin)


def _run_plugin(st):
    st.sim.pres.data[...] = 0.0
    st.solver.solve(st.sim.tmp, st.sim.pres)
    return st.sim.pres.data


def _prepare_pstep(case, seed):
    m = _mesh(case)
    p = _pressure(m, seed)
    # the last step's pressure: the new one's bulk with other small scales
    old = 0.9 * p + 0.1 * _pressure(m, seed + 1)
    rhs = _apply((m,), p)
    s = PS.Solver(**_config(case)).set_mesh(m, on_device=True)
    return SimpleNamespace(s=s, rhs=Vec(rhs), old=old, p=Vec(old.clone()), run=_run_pstep)


def _run_pstep(st):
    st.p.t.copy_(st.old)
    torch.cuda.current_stream().synchronize()
    st.s.pressure_step_device(st.rhs, st.p, rel_tol=TOL)
    return st.p.t


def _prepare_batch(case, seed):
    meshes = _batch(case)
    x = torch.cat([_pressure(m, seed * 100 + k) for k, m in enumerate(meshes)])
    b = _apply(tuple(meshes), x)
    s = PS.BatchSolver(PS.default_config(**_config(case))).set_meshes(meshes, on_device=True)
    return SimpleNamespace(s=s, b=Vec(b), x=Vec(torch.zeros_like(b)), run=_run_solve, tol=TOL)


def _prepare_operators(case, seed):
    m = _make_mesh("uniform", case["bx"], case["by"], case["px"], case["py"])
    u, v = _velocity(m, seed)
    ud, vd = _velocity(m, seed + 1)
    p = _pressure(m, seed)
    x, y, _ = _cells(m)
    lx, ly = m.domain()
    chi = torch.clamp((0.2 * min(lx, ly) - torch.hypot(x - lx / 2, y - ly / 2)) / float(m.h()[0]), 0, 1)
    # u and v go from pass to pass as from step to step; the pressure changes sign between passes, so that they stay
    # what they are in earnest however many passes there are
    return SimpleNamespace(s=PS.Solver().set_mesh(m, on_device=True), dt=_dt(m), u=Vec(u), v=Vec(v), ud=Vec(ud),
                           vd=Vec(vd), chi=Vec(chi), p=[Vec(p), Vec(-p)], rhs=Vec(torch.zeros_like(u)), run=_run_operators)


UINF, NU = (0.2, 0.05), 1e-4


def _dt(m):
    h = float(m.h()[0])
    return 0.05 * h / (NU / h + 1.0)


def _run_operators(st):
    st.s.advect_diffuse_device(st.u, st.v, UINF, NU, st.dt)
    st.s.pressure_rhs_device(st.u, st.v, st.ud, st.vd, st.chi, st.dt, st.rhs)
    st.s.pressure_correct_device(st.p[0], st.dt, st.u, st.v)
    st.p.reverse()
    return {"u": st.u.t, "v": st.v.t, "rhs": st.rhs.t}


def _prepare_step(case, seed):
    m = _make_mesh("cylinder", case["levels"], case["target"])
    fl = F.CylinderFlow(m, precision=_config(case)["precision"], rel_tol=STEP_TOL, max_iter=MAX_ITER)
    u, v = _velocity(m, seed)
    u, v = 0.2 * u - 0.1, 0.2 * v
    start = (u, v, _pressure(m, seed) * 1e-3)
    fl.u, fl.v, fl.p = (Vec(torch.zeros_like(x)) for x in start)  # the fields, held by torch
    return SimpleNamespace(fl=fl, start=start, run=_run_step)


def _run_step(st):
    at = [d.t for d in (st.fl.u, st.fl.v, st.fl.p)]
    for to, x in zip(at, st.start):
        to.copy_(x)
    torch.cuda.current_stream().synchronize()
    st.fl.step()
    return {"u": at[0], "v": at[1], "p": at[2]}


def _prepare_adapt(case, seed):
    m = _mesh(case)
    s = PS.Solver().set_mesh(m, on_device=True)
    # the flow's structure, and with it the new mesh, is the case's; its strength and the pressure are the seed's
    u, v = (np.random.default_rng(seed).uniform(0.9, 1.1) * f for f in _velocity(m, case.get("seed", 3)))
    p = _pressure(m, seed)
    x, y, _ = _cells(m)
    chi = torch.clamp(0.5 + (0.1 - torch.hypot(x - 1.0, y - 0.5)) / 0.01, 0, 1)
    torch.cuda.synchronize()
    score = s.block_score_device(Vec(u), Vec(v), Vec(chi), 1e-30)
    # about a tenth of the blocks and the body's refined, a third tagged for compression
    return SimpleNamespace(s=s, m=m, u=Vec(u), v=Vec(v), p=Vec(p), chi=Vec(chi), rtol=float(np.quantile(score, 0.9)),
                           ctol=float(np.quantile(score, 0.33)), run=_run_adapt)


def _run_adapt(st):
    st.s.set_mesh(st.m, on_device=True)
    score = st.s.block_score_device(st.u, st.v, st.chi, st.rtol)
    tags = np.where(score > st.rtol, 1, np.where(score < st.ctol, -1, 0)).astype(np.int8)
    m2, kind, src = M.adapt(st.m, tags)
    new = [Vec(torch.empty(m2.n, dtype=torch.float64, device="cuda")) for _ in range(3)]
    st.s.transfer_device(st.m, m2, kind, src, [st.u, st.v, st.p], new)
    st.s.set_mesh(m2, on_device=True)
    return {"score": score, "u": new[0].t, "v": new[1].t, "p": new[2].t, "level": m2.level, "bx": m2.bx, "by": m2.by}


# ---------------------------------------------------------------------------
# work: what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "operators":
        n = 64 * case["bx"] * case["by"]
        # u, v, ud, vd, chi, p in; u, v, rhs out; two WENO5 stages of about 400 operations per cell each
        return {"bytes": 72.0 * n, "flops": 900.0 * n}
    if kind == "adapt":
        nb = _mesh(case).n_blocks
        return {"bytes": nb * (64 * 8 * 7.0 + 200), "flops": nb * 64 * 40.0}
    blocks = [m.n_blocks for m in _batch(case)] if kind == "batch" else \
        [(_make_mesh("cylinder", case["levels"], case["target"]) if kind == "step" else _mesh(case)).n_blocks]
    # b in, x out (a step: u, v, p in and out, chi in); an iteration applies the 64 x 64 block inverse and the
    # 5-point operator twice each and updates the vectors; about 16 sqrt(blocks) of them to 1e-12
    per = 2 * (2 * 64 * 64 + 64 * 9) + 64 * 24
    return {"bytes": sum(blocks) * 64 * (56.0 if kind == "step" else 24.0 if kind == "pstep" else 16.0),
            "flops": float(sum(16 * math.sqrt(nb) * nb * per for nb in blocks))}


# ---------------------------------------------------------------------------
# exact: the same in 64 bits, by torch alone
# ---------------------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "plugin"):
        x = _pressure(_mesh(case), seed)
        return x.reshape(-1, 8, 8).cpu().numpy() if kind == "plugin" else x
    if kind == "batch":
        return torch.cat([_pressure(m, seed * 100 + k) for k, m in enumerate(_batch(case))])
    if kind == "pstep":
        m = _mesh(case)
        old = 0.9 * _pressure(m, seed) + 0.1 * _pressure(m, seed + 1)
        # p_old plus a mean-free increment
        h2 = _cells(m)[2]
        return _pressure(m, seed) + (old * h2).sum() / h2.sum()
    if kind == "operators":
        return _exact_operators(case, seed)
    return None  # whole steps on refined meshes: no plain form of that length


def _grid(m, f):
    """Block-major values as rows y, columns x."""
    g = torch.empty(m.bpdy, 8, m.bpdx, 8, dtype=f.dtype, device=f.device)
    by, bx = torch.from_numpy(m.by).long().cuda(), torch.from_numpy(m.bx).long().cuda()
    g[by, :, bx, :] = f.reshape(-1, 8, 8)
    return g.reshape(m.bpdy * 8, m.bpdx * 8)


def _blocks(m, g):
    by, bx = torch.from_numpy(m.by).long().cuda(), torch.from_numpy(m.bx).long().cuda()
    return g.reshape(m.bpdy, 8, m.bpdx, 8)[by, :, bx, :].reshape(-1)


def _pad(m, g, sx, sy, d):
    """d ghost layers: periodic, or the boundary cell times sx (x faces) or sy (y faces)."""
    x0, x1 = (g[:, -d:], g[:, :d]) if m.periodic_x else (sx * g[:, :1].expand(-1, d), sx * g[:, -1:].expand(-1, d))
    g = torch.cat([x0, g, x1], 1)
    y0, y1 = (g[-d:], g[:d]) if m.periodic_y else (sy * g[:1].expand(d, -1), sy * g[-1:].expand(d, -1))
    return torch.cat([y0, g, y1], 0)


def _weno(a, b, c, d, e, plus):
    """The fifth-order value right (plus) or left of the middle one."""
    b1 = 13 / 12 * (a + c - 2 * b) ** 2 + 0.25 * (a + 3 * c - 4 * b) ** 2
    b2 = 13 / 12 * (b + d - 2 * c) ** 2 + 0.25 * (b - d) ** 2
    b3 = 13 / 12 * (c + e - 2 * d) ** 2 + 0.25 * (3 * c + e - 4 * d) ** 2
    g1, g3 = (0.1, 0.3) if plus else (0.3, 0.1)
    w1, w2, w3 = g1 / (b1 + 1e-6) ** 2, 0.6 / (b2 + 1e-6) ** 2, g3 / (b3 + 1e-6) ** 2
    if plus:
        f1, f2, f3 = (2 * a - 7 * b + 11 * c) / 6, (-b + 5 * c + 2 * d) / 6, (2 * c + 5 * d - e) / 6
    else:
        f1, f2, f3 = (-a + 5 * b + 2 * c) / 6, (2 * b + 5 * c - d) / 6, (11 * c - 7 * d + 2 * e) / 6
    return (w1 * f1 + w2 * f2 + w3 * f3) / (w1 + w2 + w3)


def _derivative(wind, s):
    up = _weno(*s[1:6], True) - _weno(*s[0:5], True)
    return torch.where(wind > 0, up, _weno(*s[2:7], False) - _weno(*s[1:6], False))


def _advection(m, u, v, h, dt):
    ny, nx = u.shape
    U, V = u + UINF[0], v + UINF[1]
    out = []
    for f, sx, sy in ((u, -1.0, 1.0), (v, 1.0, -1.0)):
        g = _pad(m, f, sx, sy, 3)
        xs = [g[3:3 + ny, k:k + nx] for k in range(7)]
        ys = [g[k:k + ny, 3:3 + nx] for k in range(7)]
        lap = xs[2] + xs[4] + ys[2] + ys[4] - 4 * f
        out.append((-dt * h * (U * _derivative(U, xs) + V * _derivative(V, ys)) + NU * dt * lap) / h**2)
    return out


def _exact_operators(case, seed):
    m = _make_mesh("uniform", case["bx"], case["by"], case["px"], case["py"])
    h, dt = float(m.h()[0]), _dt(m)
    u, v = (_grid(m, f) for f in _velocity(m, seed))
    ud, vd = (_grid(m, f) for f in _velocity(m, seed + 1))
    p = _grid(m, _pressure(m, seed))
    x, y, _ = _cells(m)
    lx, ly = m.domain()
    chi = _grid(m, torch.clamp((0.2 * min(lx, ly) - torch.hypot(x - lx / 2, y - ly / 2)) / h, 0, 1))
    a = _advection(m, u, v, h, dt)
    a = _advection(m, u + 0.5 * a[0], v + 0.5 * a[1], h, dt)
    u, v = u + a[0], v + a[1]

    def diff(f, sx, sy):
        g = _pad(m, f, sx, sy, 1)
        return g[1:-1, 2:] - g[1:-1, :-2], g[2:, 1:-1] - g[:-2, 1:-1]

    def div(a, b):
        return diff(a, -1.0, 1.0)[0] + diff(b, 1.0, -1.0)[1]

    rhs = 0.5 * h / dt * (div(u, v) - chi * div(ud, vd))
    px, py = diff(p, 1.0, 1.0)
    return {"u": _blocks(m, u - 0.5 * dt / h * px), "v": _blocks(m, v - 0.5 * dt / h * py), "rhs": _blocks(m, rhs)}
