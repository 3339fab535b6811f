"""The launch-per-kernel solves (five kernels an iteration, replayed from a graph; the batch's item kernels), which
take meshes beyond 16,384 blocks and whatever cannot run on chip: on meshes small enough for the oracle, with
cup2d_ps_set_on_chip(CHIP_OFF).

Tolerances: a converged solve's true relative residual is the 1e-10 asked for (1.05 of it: the FP64 recurrence may
drift from it that far); solved to 1e-12 it agrees with the oracle to 1e-8, the bound of the other solver tests.
After 12 iterations two summation orders of one recurrence differ by a few hundred roundings, 1e-10 of the iterate.
Graph replay, the chunk's length and the order of the work items change no bit."""

import numpy as np
import pytest

from cup2d_amd import mesh as M
from cup2d_amd import poisson as PS
from cup2d_amd import workloads as W

pytestmark = pytest.mark.gpu

MESHES = {
    "tiny_cf": lambda: M.from_blocks(2, 2, 2, 1.0, [(0, 0, 0), (0, 1, 0), (0, 1, 1), (1, 0, 2), (1, 1, 2), (1, 0, 3),
                                                    (1, 1, 3)]),
    "uniform16x8": W.uniform_16x8_mesh,
    "graded": W.graded_disk_mesh,
    "amr6_small": lambda: W.four_disk_amr6_mesh(target=3000),
    "periodic": lambda: M.graded(8, 4, 4, 2.0, [(0.1, 0.1, 0.05), (1.9, 0.9, 0.04)], [0.3, 0.15, 0.08], True, True),
}
BOTH = pytest.mark.parametrize("precision", [PS.FP64, PS.MIXED])


def _solver(m, **cfg):
    return PS.Solver(**{"max_iter": 4000, **cfg}).set_mesh(m).set_on_chip(PS.CHIP_OFF)


def _solve(s, *a, **k):
    x, st = s.solve(*a, **k)
    assert not s.on_chip()
    return x, st


@pytest.mark.parametrize("name", list(MESHES))
@pytest.mark.parametrize("norm", [PS.NORM_INF, PS.NORM_L2])
@BOTH
def test_solve_reaches_residual(oracle, name, norm, precision):
    m = MESHES[name]()
    b = W.vortex_rhs(m, 3)
    x, st = _solve(_solver(m, norm=norm, precision=precision), b, rel_tol=1e-10)
    assert st["converged"] and (precision == PS.FP64 or st["refinements"] >= 1)
    tr = oracle.true_residual(oracle.assemble(m), b, x)
    assert (tr["rel2"] if norm == PS.NORM_L2 else tr["relinf"]) <= 1.05e-10


@pytest.mark.parametrize("mc", [0, 1])
@BOTH
def test_solve_matches_oracle(oracle, mc, precision):
    m = W.graded_disk_mesh()
    A, h2 = oracle.assemble(m, mc), oracle.h2(m)
    b = W.vortex_rhs(m, 4)
    bb = b.copy()
    if mc:
        bb[A.mean_row] = 0.0
    x, st = _solve(_solver(m, norm=PS.NORM_L2, precision=precision, mean_constraint=mc), b, rel_tol=1e-12)
    assert st["converged"]
    xr, _ = oracle.bicgstab(A, bb, mean_mode=mc, h2v=h2, rel_tol=1e-13, norm="l2", max_iter=4000)
    assert np.linalg.norm(x - oracle.mean_remove(h2, xr)) <= 1e-8 * np.linalg.norm(xr)


@pytest.mark.parametrize("norm,mc", [(PS.NORM_L2, 0), (PS.NORM_INF, 0), (PS.NORM_L2, 1)])
@pytest.mark.parametrize("breakdown_tol,max_restarts", [(1e-14, 100), (0.3, 100), (0.3, 3), (0.9, 100)])
def test_iterates_and_restarts_match_the_unfused_solver(norm, mc, breakdown_tol, max_restarts):
    m = W.graded_disk_mesh()
    b = W.vortex_rhs(m, 3)
    cfg = dict(norm=norm, max_iter=12, mean_constraint=mc, breakdown_tol=breakdown_tol)
    x1, s1 = _solve(_solver(m, **cfg), b, rel_tol=1e-30, max_restarts=max_restarts)
    x2, s2 = PS.Solver(schedule=1, **cfg).set_mesh(m).solve(b, rel_tol=1e-30, max_restarts=max_restarts)
    assert (s1["iterations"], s1["restarts"]) == (s2["iterations"], s2["restarts"])
    assert s2["restarts"] >= (2 if breakdown_tol > 0.1 else 0)
    assert np.linalg.norm(x1 - x2) <= 1e-10 * np.linalg.norm(x2)


@pytest.mark.parametrize("name", ["graded", "periodic"])
@BOTH
def test_graph_and_chunk_change_no_bit(name, precision):
    m = MESHES[name]()
    b = W.vortex_rhs(m, 7)
    s = _solver(m, precision=precision)
    x, st = _solve(s, b, rel_tol=1e-10)
    assert st["converged"]
    for cfg in ({}, dict(use_graph=0), dict(chunk=5), dict(chunk=64, use_graph=0), dict(profile=1)):
        for t in (s,) if not cfg else (_solver(m, precision=precision, **cfg),):
            y, sy = _solve(t, b, rel_tol=1e-10)
            assert np.array_equal(x, y) and sy["iterations"] == st["iterations"], cfg


@BOTH
def test_pressure_step_and_mesh_change(precision):
    """A handle keeps to its path over mesh changes, and goes back on chip when told to."""
    s = PS.Solver(norm=PS.NORM_L2, max_iter=6000, precision=precision).set_on_chip(PS.CHIP_OFF)
    for m in (W.graded_disk_mesh(), W.uniform_16x8_mesh()):
        s.set_mesh(m, on_device=True)
        b, p0 = W.vortex_rhs(m, 5), np.random.default_rng(5).normal(size=m.n) * 1e-3
        p, st = s.pressure_step(b, p0, rel_tol=1e-12)
        assert st["converged"] and not s.on_chip() and st["true_rel2"] <= 2e-12
        q, st = s.set_on_chip().pressure_step(b, p0, rel_tol=1e-12)
        assert st["converged"] and s.on_chip() and st["true_rel2"] <= 2e-12
        s.set_on_chip(PS.CHIP_OFF)
    with pytest.raises(PS._lib.SolverError, match="bad mode"):
        s.set_on_chip(4)


@pytest.fixture(scope="module")
def batch():
    ms = [W.uniform_16x8_mesh(), M.uniform(4, 2, 2.0), M.uniform(1, 1, 1.0), MESHES["periodic"]()]
    ms += W.batch64_meshes(seed=7, count=3, nmin=64, nmax=600)
    return ms, [W.vortex_rhs(m, 20 + k) for k, m in enumerate(ms)]


def _batch(ms, **cfg):
    return PS.BatchSolver(PS.default_config(**{"max_iter": 4000, **cfg})).set_meshes(ms).set_on_chip(PS.CHIP_OFF)


@pytest.mark.parametrize("norm", [PS.NORM_L2, PS.NORM_INF])
@BOTH
def test_batch_reaches_residual(oracle, batch, norm, precision):
    ms, rhs = batch
    bs = _batch(ms, norm=norm, precision=precision)
    x, st = bs.solve(np.concatenate(rhs), rel_tol=1e-10)
    assert not bs.on_chip()
    for m, b, xk, sk in zip(ms, rhs, bs.split(x), st):
        assert sk["converged"]
        tr = oracle.true_residual(oracle.assemble(m), b, xk)
        assert (tr["rel2"] if norm == PS.NORM_L2 else tr["relinf"]) <= 1.05e-10


@BOTH
def test_batch_graph_and_item_order_change_no_bit(batch, precision):
    ms, rhs = batch
    b = np.concatenate(rhs)
    cfg = dict(precision=precision, norm=PS.NORM_L2, item_blocks=4)
    bs = _batch(ms, **cfg)
    x, st = bs.solve(b, rel_tol=1e-10)
    assert all(s["converged"] for s in st)
    assert np.array_equal(x, bs.solve(b, rel_tol=1e-10)[0])
    for more in (dict(use_graph=0), dict(xcd_run=1), dict(xcd_run=4), dict(xcd_run=32), dict(profile=1)):
        y, sy = _batch(ms, **cfg, **more).solve(b, rel_tol=1e-10)
        assert np.array_equal(x, y) and [s["iterations"] for s in sy] == [s["iterations"] for s in st], more


@BOTH
def test_batch_item_sizes_and_autotune(oracle, batch, precision):
    ms, rhs = batch
    b = np.concatenate(rhs)
    ref = _batch(ms, precision=precision, norm=PS.NORM_L2).set_on_chip().solve(b, rel_tol=1e-12)[0]
    tuned = _batch(ms, precision=precision, norm=PS.NORM_L2)
    tuned.autotune(tuned.device_array(b))
    for bs in [tuned] + [_batch(ms, precision=precision, norm=PS.NORM_L2, item_blocks=ib) for ib in (1, 4, 32, 256)]:
        x, st = bs.solve(b, rel_tol=1e-12)
        assert all(s["converged"] for s in st) and not bs.on_chip()
        for xk, rk in zip(bs.split(x), bs.split(ref)):
            assert np.linalg.norm(xk - rk) <= 1e-8 * np.linalg.norm(rk)
