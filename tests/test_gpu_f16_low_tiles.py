"""The fp16 projections take units of 128 weight rows where units of 256 would leave the chip idle: ragged rows, columns and
tokens around the tiles and on both sides of the line."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# tokens, K, rows: one row, the last group / wave / tile of a unit ragged, odd K blocks, and the line (140 units of 256 rows)
@pytest.mark.parametrize("T,K,N", [(65, 32, 1), (65, 33, 31), (96, 96, 33), (97, 64, 127), (128, 130, 129), (129, 2880, 257),
                                   (200, 2880, 4096), (500, 256, 4352), (520, 256, 4352), (1000, 64, 2304), (1024, 64, 2560)])
def test_projection_both_units(lib, T, K, N):
    rng = np.random.default_rng([T, K, N])
    w = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float16)
    x = rng.standard_normal((T, K)).astype(np.float32)
    out = np.full((T, N), np.nan, np.float32)
    h = lib.f16_upload(w)
    try:
        lib.check(lib.dll.csk_matmul_transpose_f16(x.ctypes.data_as(C.c_void_p), T, K, h, out.ctypes.data_as(C.c_void_p)))
    finally:
        lib.f16_free(h)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    # two fp16 terms keep 22 bits of a row's values (2^-22 of the largest for the small ones); fp32 sums of K products of
    # deviation 1 / sqrt(K) err by at most sqrt(K) 2^-24 of a sum of deviation 1, taken four times over
    assert np.max(np.abs(out - want)) <= 4 * (np.sqrt(K) * 2.0 ** -24 + 2.0 ** -20)
