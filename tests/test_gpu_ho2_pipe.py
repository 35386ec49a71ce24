"""The pipelined 2D closure sweep where its shape changes: diagonals of 1, 2 and 4 waves (64 and 65,
128 and 129 cells), fewer diagonals than wave groups, single rows and columns, and on both sides of
where the barrier walk takes over (257 cells; in FP64 129 cells of 4 moments, 800 directions of them);
every closure of up to 4 moments.  Passes against the oracle to 1e-12 (rounding of well-conditioned cell
systems), solves with FP32 sweeps to the refinement's tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,orders,schemes,fc,bc", [
    ((1, 1), (2, 2), ("DG", "DG"), True, None), ((2, 3), (2, 2), ("DG", "DD"), False, [1, 0, 0, 2 * 0]),
    ((1, 70), (1, 2), ("DD", "DG"), True, [2, 2, 0, 0]), ((70, 1), (2, 1), ("DG", "DG"), True, [0, 0, 1, 1]),
    ((64, 66), (2, 2), ("DG", "DG"), True, [1, 0, 1, 0]), ((65, 66), (2, 2), ("DD", "DD"), True, None),
    ((67, 65), (3, 2), ("DG", "DG"), False, None), ((128, 130), (2, 2), ("DG", "DG"), False, None),
    ((130, 129), (1, 1), ("DG", "DG"), True, [0, 1, 2, 2]), ((9, 40), (4, 1), ("DD", "DG"), True, None),
    ((40, 9), (1, 4), ("DG", "DD"), True, None), ((513, 514), (1, 1), ("DG", "DG"), True, None),
    ((256, 258), (2, 2), ("DG", "DG"), False, [1, 0, 0, 0]), ((258, 257), (2, 1), ("DG", "DG"), True, None),
    ((129, 131), (2, 2), ("DG", "DG"), True, None), ((131, 129), (1, 4), ("DG", "DG"), True, None)])
def test_passes(oracle, dims, orders, schemes, fc, bc):
    from radiant_hip import problems as P, solver as S
    from util import rel_err
    p = P.small_problem(2, dims=dims, G=1, L=1, quad_order=2 if max(dims) > 200 else 4, seed=61, bc=bc)
    p.dx, p.dy = p.dx * 0.3, p.dy * 0.2
    p.scheme_order, p.scheme_order_y = orders
    p.scheme, p.scheme_y = schemes
    p.full_coupling = fc
    h = S.ResidentProblem(p)
    try:
        r = np.random.default_rng(62)
        z = r.standard_normal(h.state_length())
        q = r.standard_normal((h.d.Nc, h.d.Np)) * (np.asarray(h.d.ang.pl) <= p.Lxs)
        want = oracle.transport_pass(p, 0, 0, z, q.ravel())
        e = rel_err(h.transport_pass(0, 0, q.ravel(), z), want)
        print(dims, orders, fc, bc, e, flush=True)
        assert e < 1e-12
    finally:
        h.close()


@pytest.mark.parametrize("quad_order", [18, 20])
def test_directions(oracle, quad_order):
    """648 and 800 directions on cells of 4 moments: the pipelined sweep and the walk."""
    from radiant_hip import problems as P, solver as S
    from util import rel_err
    p = P.small_problem(2, dims=(5, 6), G=1, L=1, quad_order=quad_order, seed=63)
    p.scheme, p.scheme_y, p.scheme_order, p.scheme_order_y = "DG", "DG", 2, 2
    p.sn_type = "standard"  # the Galerkin operators of such a set are singular
    h = S.ResidentProblem(p)
    try:
        assert h.d.Nd == 2 * quad_order ** 2
        r = np.random.default_rng(64)
        z = r.standard_normal(h.state_length())
        q = r.standard_normal((h.d.Nc, h.d.Np)) * (np.asarray(h.d.ang.pl) <= p.Lxs)
        assert rel_err(h.transport_pass(0, 0, q.ravel(), z), oracle.transport_pass(p, 0, 0, z, q.ravel())) < 1e-12
    finally:
        h.close()


@pytest.mark.parametrize("dims,orders,fc,quad_order", [
    ((40, 33), (2, 2), True, 4), ((65, 70), (1, 4), True, 4), ((129, 140), (2, 2), True, 2),
    ((256, 257), (3, 2), False, 2), ((257, 258), (2, 2), False, 2)])
def test_mixed(dims, orders, fc, quad_order):
    """Against the FP64 solve, whose passes the tests above hold to the oracle."""
    from radiant_hip import problems as P, solver as S
    from util import rel_err
    p = P.small_problem(2, dims=dims, G=1, L=1, quad_order=quad_order, seed=65, bc=[1, 0, 0, 0], tol=1e-10)
    p.scheme, p.scheme_y = "DG", "DG"
    p.scheme_order, p.scheme_order_y = orders
    p.full_coupling = fc
    ref, _ = S.compute_flux(p)
    phi, st = S.compute_flux(p, precision="mixed-fp32", state="reduced")
    print(dims, orders, fc, rel_err(phi, ref), flush=True)
    assert st[0]["converged"] and st[0]["passes_lo"] > 0 and rel_err(phi, ref) < 1e-8
