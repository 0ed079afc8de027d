"""The grouped GEMM walks K in steps of four blocks, four steps to a fetch of scale bytes: every number of steps left over, on
both projections, in tiles of up to 32 tokens, of more, and of 512 weight rows.  Every weight block of a row has a scale byte
of its own (ten binades apart), so that a byte taken from a neighbouring step, block or row shows."""
import numpy as np
import pytest

from coalsack_amd import synth
from tests.helpers import assert_layer_close, build_layer, oracle_layer_subset

pytestmark = pytest.mark.gpu


def spread_scales(L, n=10):
    """The layer's own codes under n different scale bytes, small enough for outputs of order 1."""
    def blocks(e, which, plain=L.blocks):
        rows, K = (L.H, L.F) if which == 2 else (L.F, L.H)
        b = plain(e, which).reshape(rows, K // 32, 17).copy()
        b[:, :, 0] = 120 - n - int(np.log2(K)) // 2 + np.random.default_rng([e, which, rows, K]).integers(0, n, (rows, K // 32))
        return b.reshape(-1)
    L.blocks = blocks
    return L


BLOCKS, BATCHES = [1, 3, 4, 5, 8, 9, 12, 13, 16, 17, 21, 28, 31, 33], [(4, 90), (2, 130)]
# all of them on the grouped GEMM (tests/test_host_transfers.py holds them to it): E, k, H, F, T, weight in front
LAYERS = [(E, 1, *shape, T, 0) for nblk in BLOCKS for E, T in BATCHES for shape in ((32 * nblk, 96), (96, 32 * nblk))]


@pytest.mark.parametrize("nblk", BLOCKS)
@pytest.mark.parametrize("E,T", BATCHES)  # about 22 and 65 tokens per expert: short tiles, and full ones with a tail
@pytest.mark.parametrize("long_rows", ["gate/up", "down"])
def test_steps_left_over(lib, oracle, nblk, E, T, long_rows):
    H, F = (32 * nblk, 96) if long_rows == "gate/up" else (96, 32 * nblk)
    L = spread_scales(synth.LayerInputs(E, 1, H, F, seed=nblk))
    hidden = synth.hidden_states(T, H, seed=nblk + T)
    with build_layer(lib, L) as layer:
        got, pairs = layer.forward(hidden, want_pairs=True)
    want, wpairs = oracle_layer_subset(oracle, L, hidden, T)
    assert np.array_equal(pairs[..., 0], wpairs[..., 0])
    assert_layer_close(got, want)


@pytest.mark.parametrize("nblk", [2, 7, 16, 19, 22])
@pytest.mark.parametrize("long_rows", ["gate/up", "down"])
def test_steps_left_over_tall_tiles(lib, oracle, nblk, long_rows):
    wide, E, T = 8192, 2, 1000
    H, F = (32 * nblk, wide) if long_rows == "gate/up" else (wide, 32 * nblk)
    assert (T // 64 + E) * (wide // 256) > 2 * lib.device_info()[1]  # the condition for tiles of 512 rows
    L = spread_scales(synth.LayerInputs(E, 1, H, F, seed=nblk))
    hidden = synth.hidden_states(T, H, seed=nblk + T)
    with build_layer(lib, L) as layer:
        got, pairs = layer.forward(hidden, want_pairs=True)
    want, wpairs = oracle_layer_subset(oracle, L, hidden, 12)
    assert np.array_equal(pairs[:12, :, 0], wpairs[..., 0])
    assert_layer_close(got[:12], want)
