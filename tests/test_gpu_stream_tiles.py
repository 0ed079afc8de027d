"""Batches of token groups, on both sides of the line between the passes of four tokens and the tiles of up to 64: few experts,
which take passes at these sizes, many, whose tiles are short, full and with a tail, and every option on either."""
import numpy as np
import pytest

from coalsack_amd import capi, synth
from tests.helpers import (ROUTING_WEIGHT_TOL, assert_layer_close, build_layer, classify_index_mismatches, nbits_differ, oracle_layer,
                           oracle_layer_subset)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k,H,F,T", [(2, 1, 1024, 1024, 16), (1, 1, 96, 64, 17), (1, 1, 64, 96, 33), (1, 1, 64, 96, 64),
                                       (2, 2, 160, 64, 65), (8, 8, 128, 256, 20), (3, 1, 256, 96, 60), (64, 8, 64, 96, 40),
                                       (256, 16, 64, 64, 31), (5, 5, 32, 32, 29)])
@pytest.mark.parametrize("opts", [dict(), dict(weight_before_ffn=True, sigmoid=True), dict(act=1, norm=True)])
def test_tiles(lib, oracle, E, k, H, F, T, opts):
    opts = dict(opts)
    norm = opts.pop("norm", False)
    L = synth.LayerInputs(E, k, H, F, seed=T, with_norm=True)
    hidden = synth.hidden_states(T, H, seed=E + T)
    with build_layer(lib, L, norm=norm, **opts) as layer:
        got, pairs = layer.forward(hidden, capi.FWD_RMSNORM | capi.FWD_RESIDUAL if norm else 0, want_pairs=True)
        counts, toks = layer.last_dispatch(T)
    ids = pairs[..., 0].astype(int)
    assert np.array_equal(counts, np.bincount(ids.ravel(), minlength=E))
    off = np.concatenate([[0], np.cumsum(counts)])
    for e in range(E):
        assert np.array_equal(toks[off[e]:off[e + 1]], np.nonzero(np.any(ids == e, axis=1))[0])
    want, wpairs = oracle_layer(oracle, L, hidden, norm=norm, residual=norm, **opts)
    x = oracle.rmsnorm(hidden, L.norm_w, 1e-5) if norm else hidden
    assert classify_index_mismatches(oracle, x, L, pairs, wpairs)[0] == 0
    same = np.all(pairs[..., 0] == wpairs[..., 0], axis=1)
    assert np.max(np.abs(pairs[same, :, 1] - wpairs[same, :, 1])) <= ROUTING_WEIGHT_TOL
    assert_layer_close(got[same], want[same])


TILES = "expert_stream_kernel_tiles"
# layers whose batches take tiles (tests/test_host_transfers.py holds them to it): E, k, H, F, T, weight in front, hot experts
LAYERS = [(256, 16, 64, 64, 31, 0, 0), (160, 8, 160, 64, 40, 0, 0), (200, 16, 96, 288, 20, 0, 0), (132, 8, 288, 32, 100, 0, 0),
          (140, 4, 32, 96, 150, 0, 8), (140, 4, 96, 32, 200, 0, 8)]
WEIGHT_FIRST = [(32, 4, 2880, 2880, 24, 1, 0), (32, 4, 2880, 2880, 48, 1, 0), (64, 8, 2048, 768, 50, 1, 8)]


@pytest.mark.parametrize("E,k,H,F,T,wbf,hot", LAYERS)
@pytest.mark.parametrize("opts", [dict(), dict(sigmoid=True), dict(act=1, norm=True)])
def test_many_small_experts(lib, oracle, E, k, H, F, T, wbf, hot, opts):
    opts = dict(opts)
    norm = opts.pop("norm", False)
    L = synth.LayerInputs(E, k, H, F, seed=T, hot_experts=hot, with_norm=True)
    hidden = synth.hidden_states(T, H, seed=E + T)
    with build_layer(lib, L, norm=norm, **opts) as layer:
        got, pairs = layer.forward(hidden, capi.FWD_RMSNORM | capi.FWD_RESIDUAL if norm else 0, want_pairs=True)
        counts, _ = layer.last_dispatch(T)
    assert not hot or counts.max() > 64  # a full tile and a tail
    want, wpairs = oracle_layer(oracle, L, hidden, norm=norm, residual=norm, **opts)
    same = np.all(pairs[..., 0] == wpairs[..., 0], axis=1)
    assert same.all() or norm and same.mean() > 0.9
    assert_layer_close(got[same], want[same])


@pytest.mark.parametrize("E,k,H,F,T,wbf,hot", WEIGHT_FIRST)
@pytest.mark.parametrize("sigmoid", [False, True])
def test_weight_in_front(lib, oracle, E, k, H, F, T, wbf, hot, sigmoid):
    """The tiles' rows are gathered and scaled by a launch of their own."""
    L = synth.LayerInputs(E, k, H, F, seed=T, hot_experts=hot)
    hidden = synth.hidden_states(T, H, seed=E + T)
    opts = dict(weight_before_ffn=True, sigmoid=sigmoid)
    with build_layer(lib, L, device_weights=True, **opts) as layer:
        got, pairs = layer.forward(hidden, want_pairs=True)
    want, wpairs = oracle_layer_subset(oracle, L, hidden, T, **opts)
    assert np.array_equal(pairs[..., 0], wpairs[..., 0])
    assert_layer_close(got, want)


def test_tiles_equal_the_grouped_gemm(lib):
    """The units are the same code: a batch on the GEMM's side of the line, and half of it on the other."""
    L = synth.LayerInputs(32, 4, 2880, 2880, seed=3)
    hidden = synth.hidden_states(64, L.H, seed=4)
    with build_layer(lib, L, device_weights=True) as layer:
        whole, pairs = layer.forward(hidden, want_pairs=True)
        half, hpairs = layer.forward(hidden[:32], want_pairs=True)
    assert np.array_equal(pairs[:32, :, 0], hpairs[..., 0])
    same = np.all(pairs[:32] == hpairs, axis=(1, 2))
    assert same.sum() > 16 and nbits_differ(whole[:32][same], half[same]) == 0
