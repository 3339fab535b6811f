"""What a caller sees of the on-chip solve (csrc/team.hip) besides its solution: what a refused call leaves alone, who
solves when a launch cannot run, and solves at the same time."""

import ctypes
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from cup2d_amd import _lib
from cup2d_amd import mesh as M
from cup2d_amd import poisson as PS
from cup2d_amd import workloads as W

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("precision", [PS.FP64, PS.MIXED])
POLLS = 4096  # of a wait that is meant to end at its limit: 1 ms


@pytest.mark.parametrize("where", ["b", "x0"])
def test_refused_mixed_solve_leaves_x(where):
    """A non-finite residual is refused in mixed precision before anything is written: the initial guess stays, bit
    for bit."""
    m = W.uniform_16x8_mesh()
    s = PS.Solver(precision=PS.MIXED, norm=PS.NORM_L2, max_iter=2000).set_mesh(m, on_device=True)
    rng = np.random.default_rng(7)
    b, x0 = W.vortex_rhs(m, 2), rng.normal(size=m.n)
    (b if where == "b" else x0)[1234] = np.nan
    d_b, d_x = PS.DeviceArray.from_host(s, b), PS.DeviceArray.from_host(s, x0)
    with pytest.raises(PS._lib.SolverError, match="non-finite"):
        s.solve_device(d_b, d_x, rel_tol=1e-10)
    assert np.array_equal(d_x.numpy().view(np.int64), x0.view(np.int64))
    good = PS.DeviceArray.from_host(s, W.vortex_rhs(m, 2))
    d_x.upload(np.zeros(m.n))
    assert s.solve_device(good, d_x, rel_tol=1e-10)["converged"]


def _hand_over(precision, mode, mc=0):
    """A solve whose launch on chip does not run gives what CHIP_OFF gives, bit for bit, from the x0 it was given."""
    m = W.graded_disk_mesh()
    b, x0 = W.vortex_rhs(m, 6), np.random.default_rng(6).normal(size=m.n) * 1e-3
    s = PS.Solver(norm=PS.NORM_L2, max_iter=4000, precision=precision, mean_constraint=mc).set_mesh(m, on_device=True)
    ref, st0 = s.set_on_chip(PS.CHIP_OFF).solve(b, x0, rel_tol=1e-10)
    x, st = s.set_on_chip(mode, POLLS).solve(b, x0, rel_tol=1e-10)
    assert not s.on_chip() and st["converged"] and st["iterations"] == st0["iterations"]
    assert np.array_equal(x, ref)


def _hand_over_batch(precision, mode):
    ms = [W.uniform_16x8_mesh(), W.graded_disk_mesh(), M.uniform(1, 1, 1.0)]
    b = np.concatenate([W.vortex_rhs(m, 30 + k) for k, m in enumerate(ms)])
    x0 = np.random.default_rng(8).normal(size=b.size) * 1e-3
    s = PS.BatchSolver(PS.default_config(norm=PS.NORM_L2, max_iter=4000, precision=precision)).set_meshes(ms)
    ref, st0 = s.set_on_chip(PS.CHIP_OFF).solve(b, x0, rel_tol=1e-10)
    x, st = s.set_on_chip(mode, POLLS).solve(b, x0, rel_tol=1e-10)
    assert not s.on_chip() and all(t["converged"] for t in st)
    assert [t["iterations"] for t in st] == [t["iterations"] for t in st0]
    assert np.array_equal(x, ref)


@pytest.mark.parametrize("mc", [0, 1])
@BOTH
def test_short_launch_is_solved_per_kernel(precision, mc):
    _hand_over(precision, PS.CHIP_SHORT, mc)


@BOTH
def test_short_batch_launch_is_solved_per_kernel(precision):
    _hand_over_batch(precision, PS.CHIP_SHORT)


@pytest.mark.parametrize("mc", [0, 1])
@BOTH
def test_refused_launch_is_solved_per_kernel(precision, mc):
    _hand_over(precision, PS.CHIP_REFUSED, mc)


@BOTH
def test_refused_batch_launch_is_solved_per_kernel(precision):
    _hand_over_batch(precision, PS.CHIP_REFUSED)


def test_refused_noalloc_launch_is_solved_per_kernel():
    m = W.uniform_16x8_mesh()
    s = PS.Solver(norm=PS.NORM_L2, max_iter=4000).set_mesh(m, on_device=True).set_on_chip(PS.CHIP_REFUSED)
    d_b = PS.DeviceArray.from_host(s, W.vortex_rhs(m, 2))
    d_x, d_y = (PS.DeviceArray.from_host(s, np.zeros(m.n)) for _ in range(2))
    st = _lib.Stats()
    assert _lib.load().cup2d_ps_solve_device_noalloc(s.h, d_b.ptr, d_x.ptr, 0.0, 1e-10, 100, ctypes.byref(st)) == 0
    assert st.converged and not s.on_chip()
    s.set_on_chip(PS.CHIP_OFF).solve_device(d_b, d_y, rel_tol=1e-10)
    assert np.array_equal(d_x.numpy(), d_y.numpy())


@pytest.mark.parametrize("mode", [PS.CHIP_SHORT, PS.CHIP_REFUSED])
def test_a_launch_that_cannot_run_is_not_the_last(mode):
    """After a launch that could not run the next solve takes the kernels, and then the chip is tried again, after
    twice as many solves each time it fails; a mesh change tries it at once."""
    m = W.graded_disk_mesh()
    b = W.vortex_rhs(m, 6)
    s = PS.Solver(norm=PS.NORM_L2, max_iter=4000).set_mesh(m)
    bs = PS.BatchSolver(PS.default_config(norm=PS.NORM_L2, max_iter=4000)).set_meshes([m])

    def on_chip(h, mode=PS.CHIP_AUTO):
        h.set_on_chip(mode, POLLS).solve(b, rel_tol=1e-10)
        return h.on_chip()

    for h in (s, bs):
        assert not on_chip(h, mode)
        assert [on_chip(h) for _ in range(3)] == [False, True, True]
        assert not on_chip(h, mode) and not on_chip(h) and not on_chip(h, mode)
        assert [on_chip(h) for _ in range(3)] == [False, False, True]
    assert not on_chip(s, mode) and not on_chip(bs, mode)
    s.set_mesh(m, on_device=True)
    bs.set_meshes([m], on_device=True)
    assert on_chip(s) and on_chip(bs)


def test_a_team_waits_for_the_solves_before_it():
    """The first instance takes 200 of 256 workgroups for 3000 iterations, 50 ms; the others take tickets of the second,
    which has 100, and wait for the rest however short the wait for a team is set (4096 polls: 1 ms)."""
    ms = [M.uniform(128, 100, 16.0), M.uniform(80, 80, 10.0), M.uniform(16, 8, 2.0)]
    s = PS.BatchSolver(PS.default_config(norm=PS.NORM_L2, max_iter=3000)).set_meshes(ms, on_device=True)
    b = np.concatenate([W.vortex_rhs(m, k) for k, m in enumerate(ms)])
    ref = s.solve(b, rel_tol=1e-30)[0]
    assert s.on_chip()
    x = s.set_on_chip(PS.CHIP_AUTO, POLLS).solve(b, rel_tol=1e-30)[0]
    assert s.on_chip() and np.array_equal(x, ref)


@pytest.mark.parametrize("precision,mc", [(PS.MIXED, 0), (PS.MIXED, 1), (PS.FP64, 1), (PS.FP64, 0)])
@pytest.mark.parametrize("norm", [PS.NORM_L2, PS.NORM_INF])
def test_converging_in_the_last_iteration_allowed(precision, mc, norm):
    """Where convergence is confirmed on the residual, that is done after the last iteration too."""
    m = W.graded_disk_mesh()
    b = W.vortex_rhs(m, 6)
    cfg = dict(norm=norm, precision=precision, mean_constraint=mc)
    x, st = PS.Solver(max_iter=4000, **cfg).set_mesh(m).solve(b, rel_tol=1e-6)
    assert st["converged"]
    y, sy = PS.Solver(max_iter=st["iterations"], **cfg).set_mesh(m).solve(b, rel_tol=1e-6)
    assert sy["converged"] and sy["iterations"] == st["iterations"] and np.array_equal(x, y)


def test_mixed_solve_recomputes_the_residual_at_its_end():
    m = W.graded_disk_mesh()
    b = W.vortex_rhs(m, 6)
    for mode in (PS.CHIP_OFF, PS.CHIP_AUTO):
        s = PS.Solver(norm=PS.NORM_L2, precision=PS.MIXED, max_iter=25).set_mesh(m).set_on_chip(mode)
        x, st = s.solve(b, rel_tol=1e-10)
        assert st["iterations"] == 25 and not st["converged"] and st["refinements"] >= 1
        assert abs(st["err_final"] - st["true_rel2"] * np.linalg.norm(b)) <= 1e-9 * st["err_final"]


@pytest.mark.parametrize("breakdown_tol,max_restarts", [(1e-2, 20), (1e-6, 5), (1e-8, 2)])
def test_mixed_restarts_are_counted_by_pass(breakdown_tol, max_restarts):
    """A mixed solve that has used up its restarts recomputes the residual and goes on (64 passes at most), on chip as
    by launches per kernel."""
    m = W.graded_disk_mesh()
    b = W.vortex_rhs(m, 3)
    for mode in (PS.CHIP_OFF, PS.CHIP_AUTO):
        s = PS.Solver(norm=PS.NORM_L2, precision=PS.MIXED, breakdown_tol=breakdown_tol, max_iter=4000).set_mesh(m)
        x, st = s.set_on_chip(mode).solve(b, rel_tol=1e-10, max_restarts=max_restarts)
        assert st["restarts"] > max_restarts
        assert st["refinements"] == 64 or (st["converged"] and st["true_rel2"] <= 1.05e-10)


def _free():
    """Free bytes of the device, by the HIP runtime that the library has loaded."""
    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("precision,bound", [(PS.FP64, 96), (PS.MIXED, 68)])
def test_batch_memory(precision, bound):
    """Device memory per unknown: b, x, the best iterate, the host interface's copy and seven Krylov vectors (8 or 4
    bytes), and the operator (1-2 bytes on a uniform mesh)."""
    ms = [M.uniform(128, 128, 16.0)] * 16
    s = PS.BatchSolver(PS.default_config(precision=precision))
    free = _free()
    s.set_meshes(ms)
    assert free - _free() <= bound * s.n


def test_x0_of_marker_words():
    """x0 may hold any word, also the NaN that marks halo words which have not arrived."""
    m = W.uniform_16x8_mesh()
    x0 = np.full(m.n, 0x7ff4c2d0a11c0de5, np.uint64).view(np.float64)
    s = PS.Solver(norm=PS.NORM_L2, max_iter=50).set_mesh(m)
    x, st = s.solve(W.vortex_rhs(m, 2), x0, rel_tol=1e-10)
    assert s.on_chip() and not st["converged"]


@pytest.mark.parametrize("rel_tol", [1e-13, 1e-14, 1e-15])
def test_mean_row_below_the_attainable_residual(rel_tol):
    """FP64 convergence is the recurrence's (as BiCGSTAB.cu:572-593), also where rounding keeps the residual itself
    from following: on chip as by launches per kernel, and with no larger residual there."""
    for m in (W.uniform_16x8_mesh(), W.graded_disk_mesh(), W.batch64_meshes()[0]):
        b = W.vortex_rhs(m, 3)
        st = [PS.Solver(norm=PS.NORM_L2, mean_constraint=1, max_iter=4000).set_mesh(m, on_device=True)
              .set_on_chip(mode).solve(b, rel_tol=rel_tol)[1] for mode in (PS.CHIP_OFF, PS.CHIP_AUTO)]
        assert st[0]["converged"] and st[1]["converged"]
        assert st[1]["true_rel2"] <= st[0]["true_rel2"]


def test_solves_at_the_same_time():
    """Handles on threads of their own, on chip and not, a batch among them: what each gives alone."""
    ms = [M.uniform(16, 8, 2.0), M.uniform(128, 96, 16.0), W.graded_disk_mesh(), M.uniform(91, 90, 12.0)]

    def single(k, mode=PS.CHIP_AUTO):
        s = PS.Solver(norm=PS.NORM_L2, max_iter=300).set_mesh(ms[k], on_device=True).set_on_chip(mode)
        b = W.vortex_rhs(ms[k], k)
        return lambda: (s.solve(b, rel_tol=1e-30)[0], s.on_chip())

    def batch():
        s = PS.BatchSolver(PS.default_config(norm=PS.NORM_L2, max_iter=300)).set_meshes(ms)
        b = np.concatenate([W.vortex_rhs(m, k) for k, m in enumerate(ms)])
        return lambda: (s.solve(b, rel_tol=1e-30)[0], s.on_chip())

    runs = [single(0), single(1), single(2), single(3, PS.CHIP_OFF), batch()]
    alone = [run() for run in runs]
    assert [c for _, c in alone] == [True, True, True, False, True]
    wrong = []

    def work(k):
        for _ in range(6):
            x, chip = runs[k]()
            if not np.array_equal(x, alone[k][0]) or chip != alone[k][1]:
                wrong.append((k, chip))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(runs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


PROCESS = """
import numpy as np
from cup2d_amd import mesh as M, poisson as PS, workloads as W
bx, by = %d, %d
m = M.uniform(bx, by, extent=max(bx, by) / 8.0)
s = PS.Solver(norm=PS.NORM_L2, max_iter=4000).set_mesh(m, on_device=True)
b = W.vortex_rhs(m, 1)
for k in range(20):
    x, st = s.solve(b, rel_tol=1e-10)
    assert st["converged"] and st["true_rel2"] <= 1.05e-10, st
print("solved")
"""


def test_processes_at_the_same_time():
    """The runtime may refuse a process's launches on chip while another one has them (an error of state): its solves
    run by launches per kernel then."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    ps = [subprocess.Popen([sys.executable, "-c", PROCESS % g], cwd=root, stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, text=True) for g in ((16, 8), (64, 64), (91, 90), (128, 96))]
    out = [p.communicate(timeout=100)[0] for p in ps]
    assert all(p.returncode == 0 and "solved" in o for p, o in zip(ps, out)), out
