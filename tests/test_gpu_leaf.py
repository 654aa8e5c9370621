"""The panel leaf (rpanel.hip) at the sizes where its plan changes: one
workgroup with 1, 2 or 4 rows per thread (256, 512, 1024 rows), several
workgroups (real types from 1025 rows with 2 rows per thread, complex ones from
513 with 1, by the number of records a wave polls; beyond 32 workgroups of 2
rows per thread with 2 or 4), sub-panels of 16 (complex: 8) columns and ragged
last ones.

A matrix of at most 64 columns is one leaf, whose operations are those of
getrf_row_major (src/lapack/getrf.rs:55-117) in the same order, so pivots and
factors have to equal the oracle's bit for bit; no tolerance is involved.
"""
import ctypes

import numpy as np
import pytest

import lair_amd as L
from lair_amd import inputs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (15, 16), (16, 15), (17, 33), (255, 64), (256, 16), (257, 17), (512, 64), (513, 31), (1023, 48),
          (1024, 64), (1025, 64), (2048, 16), (2049, 33), (4097, 40), (8193, 24), (16385, 20), (64, 300)]
ORACLE = {np.float64: O.getrf, np.float32: O.sgetrf, np.complex128: O.zgetrf, np.complex64: O.cgetrf}
TYPES = list(ORACLE)


def _same_as_oracle(a, cols):
    ref = a.copy()
    piv_o, sing_o = ORACLE[a.dtype.type](ref)
    g = a.copy()
    piv, sing = L.getrf(g)
    assert np.array_equal(piv, piv_o)
    assert sing == sing_o
    assert np.array_equal(g[:, :cols], ref[:, :cols], equal_nan=True)


def _gauss(seed, m, n, dt):
    a = inputs.gaussian_matrix(seed, m, n)
    if np.dtype(dt).kind == "c":
        a = a + 1j * inputs.gaussian_matrix(seed + 1, m, n)
    return a.astype(dt)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("shape", SHAPES)
def test_leaf_equals_oracle(shape, dt):
    m, n = shape
    _same_as_oracle(_gauss(500 + m + n, m, n, dt), min(n, 64))


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("m", [300, 700, 1500])
def test_leaf_ties_and_empty_columns(m, dt):
    """Small integers (most columns hold equal maxima, in one wave, across
    waves and across workgroups) and columns without a candidate, first and
    last in a sub-panel."""
    rng = np.random.default_rng(m)
    a = rng.integers(-2, 3, (m, 40)).astype(np.float64)
    if np.dtype(dt).kind == "c":
        a = a + 1j * rng.integers(-2, 3, (m, 40))
    a = a.astype(dt)
    for c in (0, 7, 15, 16, 31):
        a[:, c] = 0
    _same_as_oracle(a, 40)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m", [200, 1300])
def test_leaf_extreme_values(m, dt):
    """Infinities, NaN (never chosen) and subnormal entries among the candidates."""
    tiny = np.finfo(dt).smallest_subnormal
    a = _gauss(900 + m, m, 20, dt)
    a[:, 0] = 0
    a[m - 3, 0], a[5, 0], a[m // 2, 0] = 3 * tiny, 2 * tiny, -3 * tiny
    a[7, 4] = np.nan
    a[m - 1, 9] = np.inf
    _same_as_oracle(a, 20)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("m", [300, 700, 1500, 2500, 17000])
@pytest.mark.parametrize("value", [0.0, np.nan])
def test_leaf_skips_columns_without_candidate(m, value, dt):
    """Nothing is eliminated with a column of zeros or NaN, neither in its own
    sub-panel nor right of it: an infinity in its pivot row (the diagonal is
    dominant, so row c is at position c) stays the only one of its column, and
    the NaN stay in theirs."""
    a = _gauss(1200 + m, m, 64, dt)
    a[np.arange(64), np.arange(64)] += 100
    for c in (0, 5, 18):
        a[:, c] = value
        a[c, c + 20] = np.inf
    _same_as_oracle(a, 64)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("shape", [(2049, 64), (4097, 64), (8193, 64), (16385, 64), (33000, 48)])
def test_leaf_whole_blocks_beyond_sub_panels(shape, dt):
    """Whole blocks of columns right of the next sub-panel, whose update is put
    off (up to 16384 rows) or not, with every number of records a wave polls;
    33000 rows: more than 32 workgroups."""
    m, n = shape
    if dt == np.complex128 and m > 32768:
        pytest.skip("zgetrf takes at most 32768 rows")
    _same_as_oracle(_gauss(500 + m + n, m, n, dt), n)


@pytest.mark.parametrize("m", [512, 1300, 9000, 17000])
def test_leaf_of_128_fp32_columns(m):
    """The widest leaf: eight sub-panels in one launch."""
    a = _gauss(700 + m, m, 128, np.float32)
    ref = a.copy()
    piv_o, sing_o = O.sgetrf(ref)
    ctx = L.Context()
    da, dp = L.DeviceArray.from_host(a), L.DeviceArray(128, 1, np.int64)
    sing = ctypes.c_int64(-1)
    L.check(ctx.lib.lair_sgetrf_device(ctx.h, m, 128, da.ptr, 128, dp.ptr, 128, ctypes.byref(sing)), "getrf")
    piv, lu = dp.download().ravel(), da.download()
    da.free()
    dp.free()
    ctx.close()
    assert sing_o is None and sing.value == -1
    assert np.array_equal(piv, piv_o)
    assert np.array_equal(lu, ref)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("shape", [(513, 64), (769, 40), (1025, 9), (4096, 24), (8192, 33), (16384, 17), (32768, 40)])
def test_leaf_plan_edges(shape, dt):
    """The last sizes of a plan and the first of the next."""
    m, n = shape
    _same_as_oracle(_gauss(800 + m + n, m, n, dt), n)


@pytest.mark.parametrize("dt,m,n", [(np.float64, 17000, 3200), (np.float32, 17000, 200), (np.complex128, 17000, 200),
                                    (np.complex64, 17000, 200), (np.complex64, 3000, 300)])
def test_leaf_factors_do_not_depend_on_the_plan(dt, m, n, monkeypatch):
    """At most 8, 32 and 64 workgroups: 1, 2 or 4 rows per thread for the same
    rows (f64: wide enough for the trailing update to decide as well).  Each
    leaf does the same operations, so the factors are the same bits."""
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n))
    a = (a + 1j * rng.standard_normal((m, n)) if np.dtype(dt).kind == "c" else a).astype(dt)
    name = {np.float64: "d", np.float32: "s", np.complex128: "z", np.complex64: "c"}[dt]
    out = []
    for wgs in (8, 32, 64) if m <= 8192 else (32, 64):
        monkeypatch.setenv("LAIR_PANEL_MAX_WG", str(wgs))
        ctx = L.Context()
        da, dp = L.DeviceArray.from_host(a), L.DeviceArray(n, 1, np.int64)
        sing = ctypes.c_int64(-1)
        L.check(getattr(ctx.lib, f"lair_{name}getrf_device")(ctx.h, m, n, da.ptr, n, dp.ptr, 0, ctypes.byref(sing)),
                "getrf")
        out.append((dp.download(), da.download()))
        da.free()
        dp.free()
        ctx.close()
    for piv, lu in out[1:]:
        assert np.array_equal(piv, out[0][0])
        assert np.array_equal(lu, out[0][1])
