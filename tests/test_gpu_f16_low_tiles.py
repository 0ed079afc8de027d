"""The fp16 projections take units of 128 weight rows as long as no compute unit gets two of them: ragged rows, columns and
tokens around the tiles on both sides of the line, and both kinds of unit on the same tokens."""
import ctypes as C

import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import nbits_differ

pytestmark = pytest.mark.gpu


def low(lib, tokens, N):
    """Whether units of 128 rows are taken for matrices of N rows with these tokens each: the rule."""
    return sum(-(-t // 64) for t in tokens) * -(-N // 128) <= lib.device_info()[1]


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


# tokens, K, rows: one row, the last group / wave / tile of a unit ragged, odd K blocks, and up to the line (256 units on
# as many compute units)
@pytest.mark.parametrize("T,K,N", [(65, 32, 1), (65, 33, 31), (96, 96, 33), (97, 64, 127), (128, 130, 129), (129, 2880, 257),
                                   (200, 2880, 4096), (480, 256, 4096)])
def test_units_of_128_rows(lib, T, K, N):
    assert low(lib, [T], N)
    check(lib, T, K, N)


# last M tiles of 1, 32 and 33 tokens, one to seven blocks along K, last N tiles of 193, 24, 15 and 8 rows
@pytest.mark.parametrize("K", [20, 64, 96, 130, 160, 224])
@pytest.mark.parametrize("T,N", [(65, 24001), (96, 18200), (97, 18447), (129, 14600)])
def test_edges_of_units_of_256_rows(lib, T, K, N):
    assert not low(lib, [T], N)
    check(lib, T, K, N)


@pytest.mark.parametrize("T,K,N", [(480, 256, 4097), (520, 256, 4352), (1000, 64, 2304), (1024, 64, 2560)])
def test_units_of_256_rows(lib, T, K, N):
    assert not low(lib, [T], N)
    check(lib, T, K, N)


@pytest.mark.parametrize("short,long,K,N", [(480, 520, 256, 4096), (97, 640, 224, 3689)])
def test_both_kinds_give_the_same_bits(lib, short, long, K, N):
    assert low(lib, [short], N) and not low(lib, [long], N)
    w, x = inputs(long, K, N)
    assert nbits_differ(project(lib, x[:short], w), project(lib, x, w)[:short]) == 0


# layers whose routing decides: 11 M tiles and 253 units of 128 rows, and 12 and 276 where 11.1 and 256 would be expected
@pytest.mark.parametrize("E,H,T,want", [(4, 2880, 548, True), (4, 2880, 584, False)])
def test_layer_goes_by_the_tiles_that_there_are(lib, E, H, T, want):
    L = synth.LayerInputs(E, 1, H, 64, seed=3)
    hidden = synth.hidden_states(T, H, seed=4)
    with lib.layer(E, 1, H, 64, f16=True) as layer:
        layer.set_router(L.gate_w, L.gate_b)
        layer.fill_synthetic(L.seed, L.layer)
        for e in range(E):
            layer.set_expert_f16(e, None, None, None, L.b_up[e], L.b_gate[e], L.b_down[e])
        whole, pairs = layer.forward(hidden, want_pairs=True)
        try:
            lib.set_pass_tokens((T + 4) // 5)  # more than 64: the same kernel
            short, spairs = layer.forward(hidden, want_pairs=True)
        finally:
            lib.set_pass_tokens(32768)
    tokens = np.bincount(pairs[..., 0].astype(int).ravel(), minlength=E)
    assert low(lib, tokens, H) == want, tokens
    assert nbits_differ(pairs, spairs) == 0
    assert nbits_differ(whole, short) == 0
