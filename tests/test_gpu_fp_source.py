"""The Fokker-Planck source on the matrix cores at the edges of its tiles (32 moments, 128 columns, 4
moments per step): passes against the oracle to 1e-12 (FP64 sums of at most 48 terms)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd,dims,order,k", [(1, (127,), 6, 1), (1, (128,), 32, 1), (1, (129,), 34, 1), (1, (65,), 10, 2),
                                             (3, (5, 5, 6), 6, 1)])
def test_source(oracle, nd, dims, order, k):
    from radiant_hip import problems as P, solver as S
    from util import rel_err
    p = P.small_problem(nd, N=dims[0], dims=dims if nd > 1 else None, G=2, L=2, quad_order=order, seed=91)
    r = np.random.default_rng(92)
    p.csd, p.solver_type = True, "BFP"
    p.Sb, p.dE, p.T = r.uniform(0.4, 1.6, (3, p.Nmat)), r.uniform(0.5, 1.5, 2), r.uniform(0.1, 0.4, (2, p.Nmat))
    if k > 1:
        p.scheme, p.scheme_order = "DG", k
    h = S.ResidentProblem(p)
    try:
        z = r.standard_normal(h.state_length())
        q = r.standard_normal((h.d.Nc, h.d.Np)) * (np.asarray(h.d.ang.pl) <= p.Lxs)
        for mode in (0, 1):
            e = rel_err(h.transport_pass(1, mode, q.ravel(), z), oracle.transport_pass(p, 1, mode, z, q.ravel()))
            print(nd, dims, order, mode, e, flush=True)
            assert e < 1e-12
    finally:
        h.close()
