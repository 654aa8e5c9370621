"""The batched solver where its blocks, panels and size classes end: orders at
and around 16 (a register panel), 32 (a block), 64 and 128 (one, two, four
waves), matrices without a dominant diagonal (every column interchanges rows,
within and below the block), equal magnitudes, zero columns, and entries near
the end of the exponent range (where the back substitution divides instead of
multiplying by a reciprocal).

Pivots and zero-pivot columns have to equal those of the reference's row-major
LU (the oracle); the backward error |b - A x| / (|A| |x|) is within 8 n eps: n
rounded products per unknown in each of the factorization and the two
substitutions, and the growth of the pivots of a random matrix of these orders
(below 8).
"""
import numpy as np
import pytest

import lair_amd as L
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ORDERS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64, 65, 96, 127, 128, 129, 160, 191, 225, 255, 256]


def _run(As, Bs, dtype):
    ns = np.array([len(A) for A in As], np.int32)
    rs = np.array([B.shape[1] for B in Bs], np.int32)
    da = L.DeviceArray.from_host(np.concatenate([A.ravel() for A in As]).reshape(-1, 1))
    db = L.DeviceArray.from_host(np.concatenate([B.ravel() for B in Bs]).reshape(-1, 1))
    dp = L.DeviceArray(int(ns.sum()), 1, np.int64)
    di = L.DeviceArray(len(ns), 1, np.int32)
    ctx = L.Context()
    plan = L.BatchedPlan(ctx, ns, rs, da, db, dp, di, precision=0 if dtype == np.float64 else 1)
    plan.run()
    ctx.synchronize()
    lu, x, piv, info = (d.download().ravel() for d in (da, db, dp, di))
    plan.close()
    for d in (da, db, dp, di):
        d.free()
    ctx.close()
    oa, ob, op = (np.concatenate([[0], np.cumsum(k)]) for k in (ns * ns, ns * rs, ns))
    return [(lu[oa[i]:oa[i + 1]].reshape(n, n), x[ob[i]:ob[i + 1]].reshape(n, -1), piv[op[i]:op[i + 1]], info[i])
            for i, n in enumerate(ns)]


def _oracle(A):
    ref = A.copy()
    piv, sing = O.getrf(ref) if A.dtype == np.float64 else O.sgetrf(ref)
    return ref, piv, -1 if sing is None else sing


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("scale", [0, 1])
def test_orders_and_interchanges(dtype, scale):
    rng = np.random.default_rng(97)
    e = scale * (1005 if dtype == np.float64 else 110)
    As = [np.ldexp(rng.standard_normal((n, n)), e).astype(dtype) for n in ORDERS]
    Bs = [np.ldexp(rng.standard_normal((n, r)), e).astype(dtype) for n, r in zip(ORDERS, [1, 4, 5, 16] * 6)]
    eps = float(np.finfo(dtype).eps)
    for A, B, (lu, x, piv, info) in zip(As, Bs, _run(As, Bs, dtype)):
        n = len(A)
        ref, piv_o, sing_o = _oracle(A)
        assert info == sing_o == -1
        np.testing.assert_array_equal(piv, piv_o, err_msg=f"n={n}")
        a64, b64, x64 = np.ldexp(A.astype(np.float64), -e), np.ldexp(B.astype(np.float64), -e), x.astype(np.float64)
        assert np.abs(b64 - a64 @ x64).max() <= 8 * n * eps * np.abs(a64).sum(1).max() * np.abs(x64).max(), n
        # The factors reproduce the interchanged matrix (the columns of L got
        # every later interchange).
        l64, u64 = np.tril(lu.astype(np.float64), -1) + np.eye(n), np.triu(np.ldexp(lu.astype(np.float64), -e))
        pa = a64.copy()
        for i, q in enumerate(piv):
            pa[[i, q]] = pa[[q, i]]
        assert np.abs(l64 @ u64 - pa).max() <= 8 * n * eps * np.abs(a64).max(), n


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_ties_and_zero_columns(dtype):
    rng = np.random.default_rng(98)
    As, Bs = [], []
    for n in (20, 64, 100, 130, 256):
        A = rng.standard_normal((n, n)).astype(dtype)
        A[:, 0] = np.where(rng.random(n) < 0.5, 2.0, -2.0)  # equal magnitudes over every wave
        A[: n // 2, 0] = 0.5
        As.append(A)
        Z = rng.standard_normal((n, n)).astype(dtype)
        Z[:, 7] = 0.0
        Z[:, n - 3] = 0.0
        As.append(Z)
        N = rng.standard_normal((n, n)).astype(dtype)
        N[3, 0] = np.nan  # never chosen
        As.append(N)
        Bs += [rng.standard_normal((n, 2)).astype(dtype) for _ in range(3)]
    for i, (A, (lu, x, piv, info)) in enumerate(zip(As, _run(As, Bs, dtype))):
        if i % 3 == 2:
            assert piv[0] == _oracle(A)[1][0]
            continue
        _, piv_o, sing_o = _oracle(A)
        np.testing.assert_array_equal(piv, piv_o, err_msg=f"{i} n={len(A)}")
        assert info == sing_o


def _substitute(lu, piv, B):
    """getrs.rs:23-36 in the matrix's own type."""
    x, n = B.copy(), len(lu)
    for i, p in enumerate(piv):
        x[[i, p]] = x[[p, i]]
    with np.errstate(all="ignore"):
        for k in range(n):
            x[k + 1:] -= lu[k + 1:, k:k + 1] * x[k]
        for i in range(n - 1, -1, -1):
            for k in range(i + 1, n):
                x[i] -= lu[i, k] * x[k]
            x[i] /= lu[i, i]
    return x


def _same_classes(got, ref, msg):
    for f in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(f(got), f(ref), err_msg=f"{msg} {f.__name__}")


NONFINITE = [20, 40, 64, 100, 128, 200, 256]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["inf", "inf_late", "nan_column", "zero_column"])
def test_nonfinite_entries(kind, dtype):
    """An infinity in a column right of its block, and columns of zeros or NaN
    (which eliminate nothing) whose pivot row holds one: pivots, info, and which
    entries of LU and X are NaN, +inf and -inf are those of the column by column
    elimination."""
    rng = np.random.default_rng(61)
    As, Bs = [], []
    for n in NONFINITE:
        A = rng.standard_normal((n, n)).astype(dtype) + n * np.eye(n, dtype=dtype)
        c = n // 3
        if kind == "inf":
            A[5, n - 4] = np.inf
        elif kind == "inf_late":
            A[n - 3, n - 2] = -np.inf
        else:
            for c in (1, n // 3):
                A[:, c] = 0.0 if kind == "zero_column" else np.nan
                A[c, n - 2] = np.inf
        As.append(A)
        Bs.append(rng.standard_normal((n, 3)).astype(dtype))
    for A, B, (lu, x, piv, info) in zip(As, Bs, _run(As, Bs, dtype)):
        ref, piv_o, sing_o = _oracle(A)
        msg = f"{kind} n={len(A)}"
        np.testing.assert_array_equal(piv, piv_o, err_msg=msg)
        assert info == sing_o, msg
        _same_classes(lu, ref, msg)
        _same_classes(x, _substitute(ref, piv_o, B), msg)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["rhs_inf", "rhs_inf_first", "overflow", "zero_pivot"])
def test_quotients_out_of_range(kind, dtype):
    """Infinite right-hand sides, quotients that overflow and a zero pivot: the
    back substitution's results are those of divisions."""
    rng = np.random.default_rng(62)
    As, Bs = [], []
    big = dtype(np.finfo(dtype).max / 4)
    for n in NONFINITE:
        A = rng.standard_normal((n, n)).astype(dtype) + n * np.eye(n, dtype=dtype)
        B = rng.standard_normal((n, 3)).astype(dtype)
        if kind == "rhs_inf":
            B[n - 2, 1] = np.inf
        elif kind == "rhs_inf_first":
            B[0, 2] = -np.inf
        elif kind == "overflow":
            A = (0.03 * np.eye(n)).astype(dtype)
            A[0, 1:] = dtype(0.01)
            B[0, 1] = big
            B[0, 0] = -big
        else:
            A = np.triu(A)
            A[n // 2, n // 2] = 0.0
        As.append(A)
        Bs.append(B)
    for A, B, (lu, x, piv, info) in zip(As, Bs, _run(As, Bs, dtype)):
        ref, piv_o, sing_o = _oracle(A)
        msg = f"{kind} n={len(A)}"
        np.testing.assert_array_equal(piv, piv_o, err_msg=msg)
        assert info == sing_o, msg
        want = _substitute(ref, piv_o, B)
        assert not np.isfinite(want).all()
        _same_classes(lu, ref, msg)
        _same_classes(x, want, msg)


def test_config_of_the_largest_class():
    """The plan's launch shape is that of its largest systems' class: a
    workgroup for each of them."""
    rng = np.random.default_rng(63)
    ctx = L.Context()
    for ns, grid in (([40, 64, 65, 128, 129, 256, 200], 3), ([8, 128, 65, 64], 2), ([64, 1, 33], 3)):
        ns = np.array(ns, np.int32)
        rs = np.ones(len(ns), np.int32)
        da = L.DeviceArray.from_host(rng.standard_normal((int((ns * ns).sum()), 1)))
        db = L.DeviceArray.from_host(rng.standard_normal((int(ns.sum()), 1)))
        dp, di = L.DeviceArray(int(ns.sum()), 1, np.int64), L.DeviceArray(len(ns), 1, np.int32)
        plan = L.BatchedPlan(ctx, ns, rs, da, db, dp, di)
        assert plan.config()["grid"] == grid
        plan.close()
        for d in (da, db, dp, di):
            d.free()
    ctx.close()
