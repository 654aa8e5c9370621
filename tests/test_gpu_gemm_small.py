"""The small-tile update kernel (tiles of 32 x 64, a wave 16 x 32, K by chunks
of 32) where its tiles and chunks end, up to the most large tiles it takes
(128), and the ragged strips of larger updates, padded rows included.

K multiply-adds and one subtraction round once each, so every element is within
(K + 1) eps of |A| |B| plus eps |C|.
"""
import numpy as np
import pytest

import lair_amd as L
from lair_amd import _capi

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (15, 31, 17), (16, 32, 32), (17, 33, 33), (32, 64, 64), (33, 65, 96), (31, 63, 31), (65, 127, 128),
          (255, 300, 100), (2048, 1024, 64), (2049, 1024, 64), (1300, 1500, 48), (1300, 1500, 50)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_small_tiles(m, n, k, dtype):
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s).astype(dtype) for s in ((m, k), (k, n), (m, n)))
    ctx = L.Context()
    pads = (3, 5, 1)
    da, db, dc = (L.DeviceArray.from_host(x, ld=x.shape[1] + p) for x, p in zip((a, b, c), pads))
    args = (m, n, k, da.ptr, k + pads[0], db.ptr, n + pads[1], dc.ptr, n + pads[2])
    if dtype == np.float64:
        assert ctx.lib.lair_dgemm_minus_device(ctx.h, *args) == _capi.LAIR_OK
    else:
        assert ctx.lib.lair_sgemm_minus_device(ctx.h, _capi.PREC_FP32, *args) == _capi.LAIR_OK
    got = dc.download().astype(np.float64)
    for d in (da, db, dc):
        d.free()
    ctx.close()
    a, b, c = (x.astype(np.float64) for x in (a, b, c))
    eps = float(np.finfo(dtype).eps)
    bound = (k + 1) * eps * (np.abs(a) @ np.abs(b)) + eps * np.abs(c)
    assert (np.abs(got - (c - a @ b)) <= bound).all()
