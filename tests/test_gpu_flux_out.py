"""Flux copy-out: one small piece, a few and many pieces with ragged ends (pieces hold whole cells), and
both piece sizes that a test can reach (2 and 4 MiB), every value against the oracle's flux."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,G", [((3, 2, 2), 1), ((13, 11, 12), 2), ((33, 31, 30), 3), ((48, 47, 49), 4)])
def test_flux_pieces(oracle, dims, G):
    from radiant_hip import problems, solver
    from util import rel_err
    p = problems.small_problem(3, dims=dims, G=G, L=1, quad_order=4, seed=71, tol=1e-11)
    ref, _ = oracle.solve(p)
    phi, st = solver.compute_flux(p, state="reduced")
    assert phi.shape == ref.shape
    e = rel_err(phi, ref)
    print(dims, G, phi.nbytes, e, flush=True)
    assert e < 1e-9
    # every cell and moment, so that no piece is left out or misplaced
    scale = abs(ref).max(axis=2, keepdims=True)
    assert (abs(phi - ref) <= 1e-8 * scale + 1e-12).all()
