"""Which products the FP32 matrix-core kernel accepts: its launch may hold at
most 2^32 - 1 threads along a grid dimension, 2^24 - 1 blocks of 256 (what it
does not accept runs on the scalar kernel).  The library's own function, no
GPU."""
import ctypes

import pytest

from qflex_amd import capi


@pytest.fixture(scope="module")
def fits():
    f = ctypes.CDLL(capi.LIB_PATH)["_Z12qfx_f32_fitsmmm"]
    f.restype, f.argtypes = ctypes.c_bool, [ctypes.c_uint64] * 3
    return f


@pytest.mark.parametrize("m,n,k,fit", [
    (2, 1 << 30, 17, False),            # 2^24 tiles of 32 x 64
    (2, (1 << 30) - 64, 17, True),      # one less
    ((1 << 31) - 512, 2, 17, True),     # tiles of 128 x 16
    (1 << 16, 1 << 17, 64, True),       # 2^20 tiles of 128 x 64
    (300, 300, 300, True), (9, 2, 1 << 34, True), (9, 2, (1 << 34) + 1, False),
])
def test_f32_products_fit_one_grid(fits, m, n, k, fit):
    assert fits(m, n, k) is fit
