"""Flux copy-out: the pieces of every size class and way, with distinct values of which each has to
arrive at its place, into memory that holds NaN before; and whole solves beside others."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINK, ENGINE, DIRECT = 0, 1, 2
FULL = 8 << 20  # doubles of a whole chunk


# One small piece (copied by the caller), one cell, some 2 MiB pieces with a ragged end, 50 pieces of
# 4 MiB in 24 slots and 38 of 8 MiB in 12 (every slot used again), a cell's moments of just under and
# beyond a piece (the latter without the ring), one value per cell (more cells than a grid's second axis
# holds tiles); by the copy engines one piece, whole and ragged chunks of eight 8 MiB pieces, and blocks
# that hold two pieces and a rest, one, less than a whole one, and none.
@pytest.mark.parametrize("way,G,Np,Nc,chunk", [
    (LINK, 3, 5, 7, 0), (LINK, 1, 1, 1, 0), (LINK, 3, 16, 30690, 0), (LINK, 4, 30, 218461, 0),
    (LINK, 7, 31, 181003, 0), (LINK, 1024, 1023, 3, 0), (LINK, 1024, 1025, 3, 0), (LINK, 1, 1, 2500003, 0),
    (ENGINE, 3, 5, 7, FULL), (ENGINE, 1, 1, (1 << 20) + 1, FULL), (ENGINE, 4, 16, 2 * (1 << 17), FULL),
    (ENGINE, 4, 30, 218461, FULL), (ENGINE, 7, 31, 181003, FULL + 999), (ENGINE, 1024, 1023, 20, FULL),
    (ENGINE, 1, 1, 9000001, FULL), (ENGINE, 7, 31, 81003, 2250000), (ENGINE, 7, 31, 81003, 1 << 20),
    (ENGINE, 7, 31, 81003, 150000), (ENGINE, 7, 31, 31003, 1 << 17), (ENGINE, 7, 31, 31003, (1 << 17) - 1),
    (ENGINE, 1024, 1023, 20, 1024 * 1023 - 1), (ENGINE, 1024, 1025, 3, FULL), (ENGINE, 7, 31, 31003, 0),
    (DIRECT, 3, 5, 7, 0), (DIRECT, 7, 31, 81003, 0), (DIRECT, 1, 1, 4200001, 0)])
def test_pieces(way, G, Np, Nc, chunk):
    from radiant_hip import _lib
    phi = np.arange(G * Np * Nc, dtype=np.float64).reshape(G, Np, Nc)
    out = np.full((Nc, Np, G), np.nan)
    print(way, G, Np, Nc, chunk, phi.nbytes, flush=True)
    _lib.check(_lib.lib().rt_test_flux_out(way, G, Np, Nc, _lib.ptr(phi), chunk, _lib.ptr(out)))
    assert np.array_equal(out.transpose(2, 1, 0), phi)


def test_small_flux(oracle):
    """A flux of one piece, with a source in it, through the solve's own entry point."""
    from radiant_hip import problems, solver
    from util import rel_err
    p = problems.small_problem(3, dims=(3, 3, 1), G=1, L=1, quad_order=4, seed=71, tol=1e-11)
    ref, _ = oracle.solve(p)
    assert np.abs(ref).max() > 0
    phi, _ = solver.compute_flux(p, state="reduced")
    assert phi.shape == ref.shape and rel_err(phi, ref) < 1e-9


def test_beside_solves():
    """Collections beside other problems' solves (the copy engines) give the values of one alone."""
    from radiant_hip import problems as P, solver as S
    p = P.config_3d(N=40, width=4.0, G=3, L=3, quad_order=8, Nmat=3, seed=5)
    h = S.ResidentProblem(p, precision="mixed-fp32", state="reduced")
    others = [S.ResidentProblem(P.config_3d(N=24, width=2.4, G=3, L=3, quad_order=8, Nmat=3, seed=6 + i),
                                precision="mixed-fp32", state="reduced") for i in range(3)]
    stop = threading.Event()

    def work(q):
        while not stop.is_set():
            q.solve()
    th = [threading.Thread(target=work, args=(q,)) for q in others]
    try:
        h.solve()
        alone = h.flux().copy()
        assert alone.nbytes > 16 << 20 and np.abs(alone).max() > 0  # several pieces
        for t in th:
            t.start()
        for i in range(6):
            assert np.array_equal(h.flux(), alone), i
    finally:
        stop.set()
        for t in th:
            if t.is_alive():
                t.join()
        for q in others + [h]:
            q.close()
