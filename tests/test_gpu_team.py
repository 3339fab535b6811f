"""The on-chip solve (csrc/team.hip) at the edges of its work split: one
workgroup, the first and last meshes of each launch shape (16, 32, 48 and 64
blocks per workgroup, 256 workgroups), the first mesh beyond it, remainders, block
orders in which every neighbour lies in another workgroup, and explicit rows on
both sides of a workgroup's edge.

After a fixed number of iterations the iterate is compared with the one-
operation-per-launch solver's (schedule 1): the same recurrence with other
summation orders, whose difference after 12 iterations of a residual that moves
by less than 1e3 is a few hundred roundings -- 1e-10 of the iterate.  Converged
solves are checked by the oracle's residual."""

import numpy as np
import pytest

from cup2d_amd import mesh as M
from cup2d_amd import poisson as PS
from cup2d_amd import workloads as W

pytestmark = pytest.mark.gpu


def _shuffled(m, seed):
    o = np.random.default_rng(seed).permutation(m.n_blocks)
    return M.from_blocks(m.bpdx, m.bpdy, m.levels, m.extent, np.stack([m.level, m.bx, m.by], 1)[o], m.periodic_x,
                         m.periodic_y)


GRIDS = [(1, 1), (2, 1), (5, 3), (4, 4), (17, 1), (11, 3), (13, 5), (64, 64), (241, 17), (91, 90), (331, 25), (128, 96), (25, 492), (128, 128),
         (331, 50)]


@pytest.mark.parametrize("bx,by", GRIDS)
@pytest.mark.parametrize("norm", [PS.NORM_L2, PS.NORM_INF])
def test_grid_sizes_match_the_unfused_solver(bx, by, norm):
    m = M.uniform(bx, by, extent=max(bx, by) / 8.0)
    b = np.random.default_rng(bx * 1000 + by).normal(size=m.n)
    b -= b.mean()
    cfg = dict(norm=norm, max_iter=12)
    x1, s1 = PS.Solver(**cfg).set_mesh(m, on_device=True).solve(b, rel_tol=1e-30)
    x2, s2 = PS.Solver(schedule=1, **cfg).set_mesh(m).solve(b, rel_tol=1e-30)
    assert s1["iterations"] == s2["iterations"]
    assert np.linalg.norm(x1 - x2) <= 1e-10 * np.linalg.norm(x2)


MESHES = {
    "shuffled grid": lambda: _shuffled(M.uniform(96, 90, extent=12.0), 1),
    "shuffled periodic grid": lambda: _shuffled(M.uniform(9, 7, 1.0, True, True), 2),
    "graded": W.graded_disk_mesh,
    "shuffled graded": lambda: _shuffled(W.graded_disk_mesh(), 3),
    "amr6": lambda: W.four_disk_amr6_mesh(target=5000),
    "shuffled amr6": lambda: _shuffled(W.four_disk_amr6_mesh(target=9000), 4),
    "periodic": lambda: M.graded(8, 4, 4, 2.0, [(0.1, 0.1, 0.05), (1.9, 0.9, 0.04)], [0.3, 0.15, 0.08], True, True),
}


@pytest.mark.parametrize("name", list(MESHES))
@pytest.mark.parametrize("mc", [0, 1])
def test_block_orders_and_coarse_fine_rows(oracle, name, mc):
    m = MESHES[name]()
    b = W.vortex_rhs(m, 5)
    cfg = dict(norm=PS.NORM_L2, max_iter=12, mean_constraint=mc)
    x1, s1 = PS.Solver(**cfg).set_mesh(m, on_device=True).solve(b, rel_tol=1e-30)
    x2, s2 = PS.Solver(schedule=1, **cfg).set_mesh(m).solve(b, rel_tol=1e-30)
    assert s1["iterations"] == s2["iterations"] == 12
    assert np.linalg.norm(x1 - x2) <= 1e-10 * np.linalg.norm(x2)
    A = oracle.assemble(m, mc)
    bm = b.copy()
    if mc:
        bm[A.mean_row] = 0.0
    tr = oracle.true_residual(A, bm, x1, mean_mode=mc, h2v=oracle.h2(m))
    assert abs(tr["rel2"] - s1["true_rel2"]) <= 1e-9 * tr["rel2"]


@pytest.mark.parametrize("norm,mc", [(PS.NORM_L2, 0), (PS.NORM_INF, 0), (PS.NORM_L2, 1)])
@pytest.mark.parametrize("max_iter,breakdown_tol,max_restarts", [(1, 1e-14, 100), (2, 1e-14, 100), (3, 1e-14, 100),
                                                                 (12, 0.3, 100), (12, 0.3, 3), (12, 0.9, 100)])
def test_last_iterations_and_restarts(norm, mc, max_iter, breakdown_tol, max_restarts):
    """An iteration is assessed when the next one's first sums arrive: the last one, and those that restart (a large
    breakdown tolerance: nearly all), end as the one-operation-per-launch solver's do."""
    m = W.graded_disk_mesh()
    b = W.vortex_rhs(m, 3)
    cfg = dict(norm=norm, max_iter=max_iter, mean_constraint=mc, breakdown_tol=breakdown_tol)
    x1, s1 = PS.Solver(**cfg).set_mesh(m, on_device=True).solve(b, rel_tol=1e-30, max_restarts=max_restarts)
    x2, s2 = PS.Solver(schedule=1, **cfg).set_mesh(m).solve(b, rel_tol=1e-30, max_restarts=max_restarts)
    assert (s1["iterations"], s1["restarts"]) == (s2["iterations"], s2["restarts"])
    assert s2["restarts"] >= (2 if breakdown_tol > 0.1 else 0)
    assert np.linalg.norm(x1 - x2) <= 1e-10 * np.linalg.norm(x2)
    assert abs(s1["err_final"] - s2["err_final"]) <= 1e-10 * s2["err_final"]


@pytest.mark.parametrize("precision", [PS.FP64, PS.MIXED])
def test_initial_guess_zero_rhs_and_nan(oracle, precision):
    m = W.uniform_16x8_mesh()
    s = PS.Solver(norm=PS.NORM_L2, max_iter=2000, precision=precision).set_mesh(m, on_device=True)
    b = W.vortex_rhs(m, 2)
    x, st = s.solve(b, rel_tol=1e-12)
    # from the solution itself: nothing to gain, the same (mean-free) solution returned
    y, st2 = s.solve(b, x, tol=2.0 * st["err_final"] + 1e-13, max_restarts=5)
    assert st2["converged"] or precision == PS.FP64
    assert np.linalg.norm(x - y) <= 1e-10 * np.linalg.norm(x)
    z, st3 = s.solve(np.zeros(m.n), np.full(m.n, 2.0), rel_tol=1e-10)
    assert st3["iterations"] == 0 and np.abs(z).max() <= 1e-14
    b[7] = np.nan  # every workgroup leaves
    if precision == PS.MIXED:
        with pytest.raises(PS._lib.SolverError, match="non-finite"):
            s.solve(b, rel_tol=1e-10)
    else:
        assert not s.solve(b, rel_tol=1e-10)[1]["converged"]
    assert s.solve(W.vortex_rhs(m, 2), rel_tol=1e-10)[1]["converged"]
