"""The pipelined 2D closure sweep where its shape changes: diagonals of 1, 2 and 4 waves (64 and 65,
128 and 129 cells), fewer diagonals than wave groups, single rows and columns, and the grid beyond its
diagonals that the barrier walk takes (513); every closure of up to 4 moments.  Passes against the
oracle to 1e-12 (rounding of well-conditioned cell systems)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,orders,schemes,fc,bc", [
    ((1, 1), (2, 2), ("DG", "DG"), True, None), ((2, 3), (2, 2), ("DG", "DD"), False, [1, 0, 0, 2 * 0]),
    ((1, 70), (1, 2), ("DD", "DG"), True, [2, 2, 0, 0]), ((70, 1), (2, 1), ("DG", "DG"), True, [0, 0, 1, 1]),
    ((64, 66), (2, 2), ("DG", "DG"), True, [1, 0, 1, 0]), ((65, 66), (2, 2), ("DD", "DD"), True, None),
    ((67, 65), (3, 2), ("DG", "DG"), False, None), ((128, 130), (2, 2), ("DG", "DG"), False, None),
    ((130, 129), (1, 1), ("DG", "DG"), True, [0, 1, 2, 2]), ((9, 40), (4, 1), ("DD", "DG"), True, None),
    ((40, 9), (1, 4), ("DG", "DD"), True, None), ((513, 514), (1, 1), ("DG", "DG"), True, None)])
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
