"""The fp16 projections take units of 128 weight rows where units of 256 would leave the chip idle: ragged rows, columns and
tokens around the tiles on both sides of the line, and both kinds of unit on the same tokens."""
import ctypes as C
import math

import numpy as np
import pytest

from tests.helpers import nbits_differ

pytestmark = pytest.mark.gpu


def low(lib, T, N):
    """Whether a projection of T tokens to N values takes units of 128 rows: the rule, for one matrix."""
    units = (T / 64 + max(0.5, 1 - T / 64)) * math.ceil(N / 256)
    return 2 * units <= 1.1 * lib.device_info()[1]


def inputs(T, K, N):
    rng = np.random.default_rng([T, K, N])
    return (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float16), rng.standard_normal((T, K)).astype(np.float32)


def project(lib, x, w):
    out = np.full((len(x), len(w)), np.nan, np.float32)
    h = lib.f16_upload(w)
    try:
        lib.check(lib.dll.csk_matmul_transpose_f16(x.ctypes.data_as(C.c_void_p), *x.shape, h, out.ctypes.data_as(C.c_void_p)))
    finally:
        lib.f16_free(h)
    return out


def check(lib, T, K, N):
    w, x = inputs(T, K, N)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    # two fp16 terms keep 22 bits of a row's values (2^-22 of the largest for the small ones); fp32 sums of K products of
    # deviation 1 / sqrt(K) err by at most sqrt(K) 2^-24 of a sum of deviation 1, taken four times over
    assert np.max(np.abs(project(lib, x, w) - want)) <= 4 * (np.sqrt(K) * 2.0 ** -24 + 2.0 ** -20)


# tokens, K, rows: one row, the last group / wave / tile of a unit ragged, odd K blocks, and up to the line (140 units of 256
# rows on 256 compute units)
@pytest.mark.parametrize("T,K,N", [(65, 32, 1), (65, 33, 31), (96, 96, 33), (97, 64, 127), (128, 130, 129), (129, 2880, 257),
                                   (200, 2880, 4096), (480, 256, 4352)])
def test_units_of_128_rows(lib, T, K, N):
    assert low(lib, T, N)
    check(lib, T, K, N)


# last M tiles of 1, 32 and 33 tokens, one to seven blocks along K, last N tiles of 193, 24, 15 and 8 rows
@pytest.mark.parametrize("K", [20, 64, 96, 130, 160, 224])
@pytest.mark.parametrize("T,N", [(65, 24001), (96, 18200), (97, 18447), (129, 14600)])
def test_edges_of_units_of_256_rows(lib, T, K, N):
    assert not low(lib, T, N)
    check(lib, T, K, N)


@pytest.mark.parametrize("T,K,N", [(500, 256, 4352), (520, 256, 4352), (1000, 64, 2304), (1024, 64, 2560)])
def test_units_of_256_rows(lib, T, K, N):
    assert not low(lib, T, N)
    check(lib, T, K, N)


@pytest.mark.parametrize("short,long,K,N", [(480, 520, 256, 4352), (97, 640, 224, 3689)])
def test_both_kinds_give_the_same_bits(lib, short, long, K, N):
    assert low(lib, short, N) and not low(lib, long, N)
    w, x = inputs(long, K, N)
    assert nbits_differ(project(lib, x[:short], w), project(lib, x, w)[:short]) == 0
