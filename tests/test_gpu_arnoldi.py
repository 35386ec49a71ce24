"""Arnoldi steps of the FP64 solve at the sizes where their form changes: state lengths around the
one-workgroup limit (16 moments x N cells + 32 boundary moments: 8176, 8192, 8208), tiny ones, long
ones, and restarts around the 33 vectors the kernels hold (34: the chain of reductions).  The
iteration counts and the flux are the oracle's (both converge to 1e-12; they differ by rounding)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,restart", [(1, 30), (3, 30), (3, 2), (509, 30), (510, 30), (510, 3), (511, 30), (511, 12), (63, 33), (63, 34)])
def test_solve_forms(oracle, cells, restart):
    from radiant_hip import problems, solver
    from util import rel_err
    p = problems.small_problem(1, N=cells, G=2, L=3, quad_order=16, seed=31, tol=1e-12, bc=[1, 0])
    p.restart = restart
    ref, rst = oracle.solve(p)
    # every group has a flux and at least one Arnoldi step beside the pass that gives the residual
    assert all(np.abs(ref[g]).max() > 0 and rst[g]["niter"] > 1 for g in range(p.G))
    phi, st = solver.compute_flux(p)
    print(cells, restart, rel_err(phi, ref), [s["niter"] for s in st], [s["niter"] for s in rst], flush=True)
    assert rel_err(phi, ref) < 1e-10 and all(s["converged"] for s in st)
    assert [s["niter"] for s in st] == [s["niter"] for s in rst]


@pytest.mark.parametrize("restart", [33, 34, 40, 63])
def test_mixed_restarts(oracle, restart):
    """Inner cycles of the mixed solve that go on beyond the 33 vectors the kernels hold, where the
    restart lets them: a diffusive slab that takes more than 33 iterations to the inner tolerance."""
    from radiant_hip import problems, solver
    from util import rel_err
    p = problems.small_problem(1, N=60, G=1, L=1, quad_order=8, seed=31, tol=1e-10)
    p.sigt[:] = 2.0
    p.sigs[:] = 0.0
    p.sigs[..., 0] = 2.0 * 0.999
    p.restart = restart
    ref, _ = oracle.solve(p)
    phi, st = solver.compute_flux(p, precision="mixed-fp32", state="reduced")
    s = st[0]
    print(restart, rel_err(phi, ref), s["niter"], s["refinements"], flush=True)
    assert s["converged"] and rel_err(phi, ref) < 1e-7  # a residual of 1e-10 behind a scattering ratio of 0.999
    assert s["niter"] > 33 * s["refinements"]


@pytest.mark.parametrize("depth", [1, 2, 8, 9])
def test_anderson_depths(oracle, depth):
    """The one-pass Anderson iteration (depths up to 8) and the vector-by-vector one beyond it, on a
    solve long enough for the oldest difference to leave the history."""
    from radiant_hip import problems, solver
    from util import rel_err
    p = problems.small_problem(2, dims=(9, 7), G=2, L=2, quad_order=4, seed=33, tol=1e-11, bc=[1, 1, 0, 1])
    p.accel, p.depth = "anderson", depth
    ref, rst = oracle.solve(p)
    phi, st = solver.compute_flux(p)
    print(depth, rel_err(phi, ref), [s["niter"] for s in st], [s["niter"] for s in rst], flush=True)
    assert rel_err(phi, ref) < 1e-9 and all(s["converged"] for s in st)
    assert max(s["niter"] for s in st) > depth + 2
