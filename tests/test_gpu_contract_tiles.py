"""Work-tile sizes of the contractions (half-size tiles up to a number of them: 512 in M, 768 for up to 32
rows, 1536 in D and in M of BF16 operands): one value past and short of each tile edge, on both sides of each rule, ragged shapes
in both sizes and every operand precision, against a host product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# K products and sums, each rounded once (K eps |A||B| bounds the error); FP32 operands alike.  BF16
# operands are rounded to 8 significant bits, 2^-8 relative each (products: 2 * 2^-8 + 2^-16), and summed in
# FP32
EPS = {0: 2.0 ** -52, 1: 2.0 ** -23, 2: 2.0 ** -23}
OPERANDS = {0: 0.0, 1: 0.0, 2: 2.0 ** -7 + 2.0 ** -16}

SHAPES = [(1, 1, 1), (31, 9, 127), (33, 5, 129), (64, 35, 256), (65, 33, 257)]
M_SHAPES = [(64, 7, 256 * 128), (64, 7, 256 * 128 + 1), (63, 33, 256 * 128 - 1), (65, 33, 172 * 128 + 1),
            (32, 5, 768 * 128), (31, 9, 768 * 128 + 1)]
D_SHAPES = [(64, 7, 768 * 128), (64, 7, 768 * 128 + 1), (63, 33, 768 * 128 - 1), (65, 33, 512 * 128 + 1),
            (31, 9, 1536 * 128 + 1)]


@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("which,shape", [(0, s) for s in SHAPES + M_SHAPES] + [(1, s) for s in SHAPES + D_SHAPES] +
                         [(0, s) for s in D_SHAPES])
def test_tiles(shape, which, prec):
    from radiant_hip import _lib
    M, K, N = shape
    rng = np.random.default_rng(M + K + which)
    A, B, C = rng.standard_normal((M, K)), rng.standard_normal((K, N)), np.zeros((M, N))
    _lib.check(_lib.lib().rt_test_contraction(which, prec, M, K, N, _lib.ptr(A), _lib.ptr(B), _lib.ptr(C)))
    bound = (OPERANDS[prec] + (K + 2) * EPS[prec]) * (np.abs(A) @ np.abs(B))
    assert (np.abs(C - A @ B) <= bound).all(), (shape, which, prec, float((np.abs(C - A @ B) / bound).max()))
