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
from lair_amd import _capi, inputs

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


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n,nrhs", [(129, 1), (300, 3)])
def test_complex_getrs_waits_give_up(n, nrhs, dtype):
    """A wait limit of 0 ends the first wait of every workgroup at once: the
    call reports it, and the next call on the context solves."""
    a = (inputs.gaussian_matrix(8300 + n, n, n) + 4.0 * np.sqrt(n) * np.eye(n)).astype(dtype)
    b = inputs.gaussian_matrix(8400 + n, n, nrhs).astype(dtype)
    g = a.copy()
    piv, _ = L.getrf(g)
    ctx = L.Context()
    fn = ctx.lib.lair_zgetrs_device if dtype == np.complex128 else ctx.lib.lair_cgetrs_device
    dlu, dp, db = L.DeviceArray.from_host(g), L.DeviceArray.from_host(piv.reshape(-1, 1)), L.DeviceArray.from_host(b)
    args = (ctx.h, n, nrhs, dlu.ptr, n, dp.ptr, db.ptr, nrhs)
    L.check(ctx.lib.lair_context_set_wait_limit(ctx.h, 0), "wait limit")
    try:
        st = fn(*args)
    finally:
        L.check(ctx.lib.lair_context_set_wait_limit(ctx.h, 1 << 23), "wait limit")
    assert st == _capi.LAIR_ERR_SYNC
    db.upload(b)
    L.check(fn(*args), "getrs")
    np.testing.assert_array_equal(db.download(), L.getrs(g, piv, b))
    for d in (dlu, dp, db):
        d.free()
    ctx.close()


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
def test_complex_getrs_more_than_one_pass(dtype):
    """n=150: a pass takes 64 * 16384 / 150 = 6990 right-hand sides; the last
    ones come in a second pass.  The same right-hand sides alone (a pass of
    their own) give the same bits."""
    n, nrhs = 150, 6993
    a = (inputs.gaussian_matrix(8500, n, n) + 4.0 * np.sqrt(n) * np.eye(n)).astype(dtype)
    b = (inputs.gaussian_matrix(8501, n, nrhs) + 1j * inputs.gaussian_matrix(8502, n, nrhs)).astype(dtype)
    piv, _ = L.getrf(a)
    x = L.getrs(a, piv, b)
    for c in (0, 6989, 6990, 6992):
        assert np.array_equal(L.getrs(a, piv, b[:, c:c + 1].copy()), x[:, c:c + 1]), c


def _back_substitute(u, b):
    """x with u x = b, component by component: num-complex's product and quotient."""
    x, n = b.copy(), len(b)
    with np.errstate(all="ignore"):
        for i in range(n - 1, -1, -1):
            for k in range(i + 1, n):
                re = u[i, k].real * x[k].real - u[i, k].imag * x[k].imag
                im = u[i, k].real * x[k].imag + u[i, k].imag * x[k].real
                x.real[i] -= re
                x.imag[i] -= im
            d = u[i, i]
            ns = d.real * d.real + d.imag * d.imag
            re = (x[i].real * d.real + x[i].imag * d.imag) / ns
            im = (x[i].imag * d.real - x[i].real * d.imag) / ns
            x.real[i], x.imag[i] = re, im
    return x


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [130, 192, 300])
def test_complex_quotients_that_overflow(n, dtype):
    """A quotient that overflows is infinite, not NaN, and the rows above see
    it so: the same entries are NaN, +inf and -inf as with plain quotients."""
    big = np.finfo(dtype).max / 4
    u = (np.triu(np.full((n, n), 0.01)) + 0.03 * np.eye(n)).astype(dtype)
    b = (inputs.gaussian_matrix(8600, n, 3) + 1j * inputs.gaussian_matrix(8601, n, 3)).astype(dtype)
    b[0, 1] = big
    b[70, 2] = -1j * big
    want = _back_substitute(u, b)
    got = L.getrs(u, np.arange(n), b)
    assert np.isposinf(want[0, 1].real) and np.isfinite(want[:, 0]).all()
    for part in ("real", "imag"):
        for f in (np.isnan, np.isposinf, np.isneginf):
            np.testing.assert_array_equal(f(getattr(got, part)), f(getattr(want, part)), err_msg=f"{part} {f.__name__}")
