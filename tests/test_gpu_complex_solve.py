"""The dataflow complex getrs (n > 128) where its 64-row blocks end, with one,
several and more right-hand sides than one pass takes (64), and with diagonal
entries far from 1 in the exponent (the back substitution then divides directly
instead of multiplying by a corrected inverse).

The backward error |b - A x| / (|A| |x|) of every column is within 8 n eps: n
complex multiply-subtracts per unknown (each within 2 eps) in each of the
factorization and the two substitutions of a matrix whose pivots do not grow.
"""
import numpy as np
import pytest

import lair_amd as L
from lair_amd import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nrhs,scale", [(129, 1, 0), (191, 3, 0), (192, 2, 0), (193, 67, 0), (320, 1, 1), (513, 5, 1),
                                          (1025, 2, 0)])
def test_complex_getrs_blocks(n, nrhs, scale, dtype):
    def gauss(seed, k):
        return inputs.gaussian_matrix(seed, n, k) + 1j * inputs.gaussian_matrix(seed + 1, n, k)

    s = 2.0 ** (scale * (300 if dtype == np.complex128 else 40))
    a = ((gauss(8100 + n, n) + 4.0 * np.sqrt(n) * np.eye(n)) * s).astype(dtype)
    b = gauss(8200 + n, nrhs).astype(dtype)
    g = a.copy()
    piv, sing = L.getrf(g)
    assert sing is None
    x = L.getrs(g, piv, b).astype(np.complex128)
    a128 = a.astype(np.complex128)
    r = b.astype(np.complex128) - a128 @ x
    berr = np.abs(r).max(0) / (np.abs(a128).sum(1).max() * np.abs(x).max(0))
    assert berr.max() <= 8 * n * float(np.finfo(dtype).eps)
