"""The scanned 1D slowing-down sweep at the edges of its steps (64 lanes of 2 cells up to 4 moments
per cell, of 1 beyond): passes against the oracle's cell-by-cell sweep to 1e-12 (rounding of affine
maps whose factors stay below 1), one and several steps, reflective and periodic faces, every cell
form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,orders,schemes,fc,bc", [
    (1, (2, 2), ("DG", "DG"), True, None), (127, (2, 2), ("DG", "DG"), True, [1, 0]),
    (128, (2, 2), ("DD", "DG"), False, [2, 2]), (129, (1, 4), ("DD", "DG"), True, None),
    (300, (2, 1), ("DG", "DD"), True, [1, 1]), (63, (2, 3), ("DG", "DD"), True, [0, 1]),
    (64, (2, 4), ("DG", "DG"), True, None), (65, (2, 4), ("DD", "DD"), False, [1, 0]),
    (130, (1, 3), ("DG", "DG"), True, None)])
def test_passes(oracle, cells, orders, schemes, fc, bc):
    from radiant_hip import problems as P, solver as S
    from util import rel_err
    p = P.small_problem(1, N=cells, G=2, L=2, quad_order=6, seed=51, bc=bc)
    r = np.random.default_rng(52)
    p.csd, p.Sb, p.dE = True, r.uniform(0.4, 1.6, (3, p.Nmat)), r.uniform(0.5, 1.5, 2)
    p.scheme_order_e, p.scheme_order = orders
    p.scheme_e, p.scheme = schemes
    p.full_coupling = fc
    h = S.ResidentProblem(p)
    try:
        z = r.standard_normal(h.state_length())
        q = r.standard_normal((h.d.Nc, h.d.Np)) * (np.asarray(h.d.ang.pl) <= p.Lxs)
        for mode in (0, 1):
            want = oracle.transport_pass(p, 1, mode, z, q.ravel())
            e = rel_err(h.transport_pass(1, mode, q.ravel(), z), want)
            print(cells, orders, fc, bc, mode, e, flush=True)
            assert e < 1e-12
    finally:
        h.close()
    if cells < 130:
        p.tol = 1e-12
        ref, _ = oracle.solve(p)
        for prec, tol in (("fp64", 1e-10), ("mixed-fp32", 1e-6)):
            phi, st = S.compute_flux(p, precision=prec, state="faithful" if prec == "fp64" else "reduced")
            assert rel_err(phi, ref) < tol and all(s["converged"] for s in st)
