"""The on-chip solve of a batch (csrc/batch.hip, plan_teams) at the edges of its
work split: one instance, exactly as many workgroups as run at once and one
more, more instances than workgroups (they start as workgroups come free),
instances of one block beside the largest, and an instance that is too large for
the chip, with which the whole batch takes the item kernels.

As for the single solve: after 12 iterations an iterate differs from the one-
operation-per-launch solver's by a few hundred roundings, 1e-10 of it."""

import numpy as np
import pytest

from cup2d_amd import mesh as M
from cup2d_amd import poisson as PS
from cup2d_amd import workloads as W

pytestmark = pytest.mark.gpu

BATCHES = {
    "one block": [(1, 1)],
    "256 workgroups of 16": [(16, 16)] * 16,
    "257 workgroups of 16": [(16, 16)] * 16 + [(1, 1)],
    "256 workgroups of 64, then one more": [(64, 64)] * 4 + [(3, 1)],
    "300 instances": [(1 + k % 5, 1 + k % 3) for k in range(300)],
    "queued": [(128, 128), (65, 1), (90, 91), (2, 2), (70, 60), (33, 30), (13, 5), (128, 128), (1, 1)],
    "too large": [(331, 50), (3, 2)],
}


@pytest.mark.parametrize("name", list(BATCHES))
@pytest.mark.parametrize("norm", [PS.NORM_L2, PS.NORM_INF])
def test_batches_match_the_unfused_solver(name, norm):
    ref = {}  # by grid: the mesh, b, the iterate
    for bx, by in set(BATCHES[name]):
        m = M.uniform(bx, by, extent=max(bx, by) / 8.0)
        b = np.random.default_rng(bx * 1000 + by).normal(size=m.n)
        b -= b.mean()
        x, st = PS.Solver(schedule=1, norm=norm, max_iter=12).set_mesh(m).solve(b, rel_tol=1e-30)
        ref[bx, by] = m, b, x, st
    parts = [ref[g] for g in BATCHES[name]]
    bs = PS.BatchSolver(PS.default_config(norm=norm, max_iter=12)).set_meshes([p[0] for p in parts])
    for _ in range(2):
        x, st = bs.solve(np.concatenate([p[1] for p in parts]), rel_tol=1e-30)
        for xk, sk, p in zip(bs.split(x), st, parts):
            assert sk["iterations"] == p[3]["iterations"]
            assert np.linalg.norm(xk - p[2]) <= 1e-10 * np.linalg.norm(p[2])


@pytest.mark.parametrize("mc", [0, 1])
def test_coarse_fine_batch(oracle, mc):
    ms = [W.graded_disk_mesh(), M.uniform(1, 1, 1.0), W.four_disk_amr6_mesh(target=5000),
          M.graded(8, 4, 4, 2.0, [(0.1, 0.1, 0.05), (1.9, 0.9, 0.04)], [0.3, 0.15, 0.08], True, True),
          W.four_disk_amr6_mesh(target=9000)]
    rhs = [W.vortex_rhs(m, 40 + k) for k, m in enumerate(ms)]
    cfg = dict(norm=PS.NORM_L2, mean_constraint=mc)
    x, st = PS.BatchSolver(PS.default_config(max_iter=12, **cfg)).set_meshes(ms).solve(np.concatenate(rhs), rel_tol=1e-30)
    off = np.concatenate([[0], np.cumsum([m.n for m in ms])])
    for k, (m, b) in enumerate(zip(ms, rhs)):
        y, s2 = PS.Solver(schedule=1, max_iter=12, **cfg).set_mesh(m).solve(b, rel_tol=1e-30)
        assert st[k]["iterations"] == s2["iterations"]
        if m.n_blocks > 1:  # one block is solved within rounding before the 12th iteration
            assert np.linalg.norm(x[off[k]:off[k + 1]] - y) <= 1e-10 * np.linalg.norm(y)
    for precision in (PS.FP64, PS.MIXED) if mc == 0 else ():
        s = PS.BatchSolver(PS.default_config(precision=precision, max_iter=6000, **cfg)).set_meshes(ms)
        x, st = s.solve(np.concatenate(rhs), rel_tol=1e-10)
        for k, (m, b, xk) in enumerate(zip(ms, rhs, s.split(x))):
            assert st[k]["converged"], (k, st[k])
            tr = oracle.true_residual(oracle.assemble(m), b, xk, mean_mode=0, h2v=oracle.h2(m))
            assert tr["rel2"] <= 1.05e-10
