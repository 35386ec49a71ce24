"""The allocation-free pass reads and writes the caller's vectors in their own layout: every form of
problem it takes gives rt_problem_pass's result bit for bit (both run the same sums in the same
order), for outputs beside the input, in place of it and overlapping it."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(form):
    from radiant_hip import problems as P
    if form == "slab1":  # one column tile, one row tile, both ragged
        return P.small_problem(1, N=5, G=2, L=3, quad_order=6, seed=1)
    if form == "slab257":  # one column past a work tile
        return P.small_problem(1, N=257, G=2, L=7, quad_order=16, seed=2)
    if form == "plane450":  # full-size tiles in M and D, the last ones ragged
        return P.small_problem(2, dims=(450, 441), G=1, L=1, quad_order=2, seed=9)
    if form == "plane130":  # full-size tiles in M, half-size in D
        return P.small_problem(2, dims=(130, 127), G=1, L=3, quad_order=8, seed=10, bc=[1, 0, 0, 1])
    if form == "plane72":  # 72 moments: a second, ragged row group
        return P.small_problem(2, dims=(17, 16), G=2, L=3, quad_order=6, seed=3)
    if form == "box48":
        return P.small_problem(3, dims=(7, 6, 9), G=2, L=2, quad_order=6, seed=4)
    if form == "reflected":
        return P.small_problem(2, dims=(13, 9), G=2, L=2, quad_order=4, seed=5, bc=[1, 0, 2, 2])
    if form == "closure":
        p = P.small_problem(2, dims=(9, 8), G=2, L=2, quad_order=4, seed=6, bc=[1, 0, 0, 1])
        p.scheme = p.scheme_y = "DG"
        p.scheme_order = p.scheme_order_y = 2
        return p
    p = P.small_problem(1, N=21, G=2, L=3, quad_order=8, seed=7)  # "fokker-planck"
    r = np.random.default_rng(8)
    p.csd, p.solver_type = True, "BFP"
    p.Sb, p.dE, p.T = r.uniform(0.5, 2, (3, 2)), r.uniform(0.5, 1.5, 2), r.uniform(0.1, 0.5, (2, 2))
    return p


@pytest.mark.parametrize("form", ["slab1", "slab257", "plane130", "plane450", "plane72", "box48", "reflected", "closure", "fokker-planck"])
def test_caller_layout_forms(form):
    from test_zz_no_alloc import _Dev
    from radiant_hip import _lib, solver
    p = _problem(form)
    h = solver.ResidentProblem(p)
    try:
        S, d = h.state_length(), h.d
        rng = np.random.default_rng(40)
        z = rng.uniform(-1.0, 1.0, S)
        q = rng.uniform(0.0, 1.0, (d.Nc, d.Np)) * (np.asarray(d.ang.pl)[None] <= p.Lxs)
        dev = _Dev()
        dq = dev.put(q.ravel())
        for g in range(p.G):
            for mode in (0, 1, 2):
                print(form, g, mode, flush=True)
                want = h.transport_pass(g, mode, q.ravel(), z)
                for shift in (None, 0, 3):  # beside the input, in place, overlapping it
                    dz = dev.put(np.concatenate([z, np.zeros(3)]))
                    out = dev.alloc(S * 8) if shift is None else C.c_void_p(dz.value + 8 * shift)
                    _lib.check(_lib.lib().rt_problem_pass_device(h.h, g, mode, dq, dz, out))
                    assert np.array_equal(dev.get(out, S), want), (form, g, mode, shift)
                    dev.free(*((dz,) if shift is not None else (dz, out)))
        dev.free(dq)
    finally:
        h.close()
