"""What a caller sees of the on-chip solve (csrc/team.hip) besides its solution: what a refused call leaves alone."""

import numpy as np
import pytest

from cup2d_amd import poisson as PS
from cup2d_amd import workloads as W

pytestmark = pytest.mark.gpu


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
