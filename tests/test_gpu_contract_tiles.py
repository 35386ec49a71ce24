"""Work-tile sizes of the contractions (half-size tiles below 512 full-size ones): one value past and
short of each tile edge, on both sides of the rule, against a host product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# FP64: K products and sums, each rounded once (K eps |A||B| bounds the error); FP32 operands alike
EPS = {0: 2.0 ** -52, 1: 2.0 ** -23}


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("shape", [(1, 1, 1), (31, 9, 127), (33, 5, 129), (64, 35, 256), (65, 33, 257),
                                   (64, 7, 511 * 256), (64, 7, 511 * 256 + 1), (63, 33, 512 * 256 - 1)])
def test_tiles(shape, which, prec):
    from radiant_hip import _lib
    M, K, N = shape
    rng = np.random.default_rng(M + K + which)
    A, B, C = rng.standard_normal((M, K)), rng.standard_normal((K, N)), np.zeros((M, N))
    _lib.check(_lib.lib().rt_test_contraction(which, prec, M, K, N, _lib.ptr(A), _lib.ptr(B), _lib.ptr(C)))
    bound = (K + 2) * EPS[prec] * (np.abs(A) @ np.abs(B))
    assert (np.abs(C - A @ B) <= bound).all(), (shape, which, prec, float((np.abs(C - A @ B) / bound).max()))
