"""The matrix-core dataflow triangular solve (trsm_mfma_kernel) where its blocks
and chunks end: ragged last row blocks (64 rows in FP64, 128 in FP32), one
element past and short of a block, partial and several chunks of 16 right-hand
sides, odd row pitches (whose tiles are not 16-byte aligned), both directions
of the solve and the transposed solve.

On A = N(0, 1) + 4 sqrt(n) I the backward error |b - A x| / (|A| |x|) of every
column is within n eps: n products per unknown, each rounded once, in the two
triangular solves and the factorization (whose pivots do not grow here).
"""
import numpy as np
import pytest

import lair_amd as L
from lair_amd import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,nrhs", [(129, 2), (191, 15), (192, 16), (193, 17), (257, 33), (640, 3), (1001, 48)])
@pytest.mark.parametrize("trans", [False, True])
def test_several_right_hand_sides(n, nrhs, trans, dtype):
    a = (inputs.gaussian_matrix(7100 + n, n, n) + 4.0 * np.sqrt(n) * np.eye(n)).astype(dtype)
    b = inputs.gaussian_matrix(7101 + n, n, nrhs).astype(dtype)
    g = a.copy()
    piv, sing = L.getrf(g)
    assert sing is None
    x = L.getrs(g, piv, b, trans=trans).astype(np.float64)
    a64 = (a.T if trans else a).astype(np.float64)
    r = b.astype(np.float64) - a64 @ x
    berr = np.abs(r).max(0) / (np.abs(a64).sum(1).max() * np.abs(x).max(0))
    assert berr.max() <= n * float(np.finfo(dtype).eps)
